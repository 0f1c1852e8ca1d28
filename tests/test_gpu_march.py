"""The marching kernels (csrc/march.hip) against the oracle, bit for bit, at
the sizes where their split can go wrong: layers narrower than a strip, one
column either side of the strip widths (60 and 56 columns) and of a wave,
layers of a few rows, a row count off every segment length, and step counts
that end on every remainder of the launches' two and four steps."""
import pytest

from gcomcot import DeviceRun
from gcomcot import scenarios as S
from helpers import compare_device_oracle, diff_report
from oracle.bind import Oracle

pytestmark = pytest.mark.gpu

SIZES = [(8, 7), (24, 5), (55, 24), (57, 33), (60, 13), (61, 40), (64, 29), (65, 26), (112, 31),
         (121, 17), (123, 50), (181, 9), (1150, 611)]


@pytest.mark.parametrize("nx,ny", SIZES, ids=[f"{a}x{b}" for a, b in SIZES])
def test_marched_layer_matches_oracle(nx, ny):
    sc = S.custom(laycord=0, laygov=0, nx=nx, ny=ny, cx=0.4)
    orc = Oracle(sc, 32, pow_mode=1)
    dev = DeviceRun(sc)
    try:
        for n, graph in [(2, True), (3, True), (4, False), (5, True), (1, True), (6, True)] + \
                ([(73, True)] if nx < 200 else [(135, True), (16, False)]):
            print(f"[gpu] march {nx}x{ny} run {n} graph={graph}", flush=True)
            dev.run(n, graph=graph)
            orc.step(n)
            compare_device_oracle(sc, dev, orc, f"march {nx}x{ny} after {n}")
    finally:
        dev.close()


@pytest.mark.parametrize("nx,ny", [(2051, 1537), (4099, 1711)], ids=["2051x1537", "4099x1711"])
def test_marched_large_layer_matches_tiles(nx, ny):
    """Layers large enough for the longer segments, against the tile kernels
    (one step per launch), which the oracle pins."""
    import numpy as np
    from gcomcot._lib import ip, lib
    sc = S.linear_layer(nx=nx, ny=ny)
    got = []
    try:
        for mode in (0, 1):
            print(f"[gpu] march {nx}x{ny} mode {mode}", flush=True)
            assert lib().gcomcot_set_temporal_blocking_(ip(mode)) == 0
            dev = DeviceRun(sc)
            dev.run(31)
            dev.run(10, graph=False)
            got.append((dev.state(1), dev.maxima(1)))
            dev.close()
    finally:
        lib().gcomcot_set_temporal_blocking_(ip(1))
    (a, am), (b, bm) = got
    for k in ("z1", "m1", "n1"):
        assert np.array_equal(a[k].view(np.int32), b[k].view(np.int32)), k
    for k in ("zmax_wet", "arrival"):
        assert np.array_equal(am[k].view(np.int32), bm[k].view(np.int32)), k


NL_SIZES = [(24, 9), (59, 30), (61, 33), (121, 47), (133, 61), (194, 59), (253, 74), (312, 45)]


@pytest.mark.parametrize("laycord", [0, 1], ids=["sph", "cart"])
@pytest.mark.parametrize("nx,ny", NL_SIZES, ids=[f"{a}x{b}" for a, b in NL_SIZES])
def test_marched_nonlinear_layer_matches_oracle(nx, ny, laycord):
    """Nonlinear layers in marching strips of every segment length, on beaches
    that flood and break: side strips, end rows and middle segments."""
    from gcomcot._lib import ip, lib
    from helpers import BEACH, surf_zone
    for sc in (S.custom(laycord=laycord, laygov=1, nx=nx, ny=ny, **BEACH),
               surf_zone(laycord, nx=nx, ny=ny)):
        orc = Oracle(sc, 32, pow_mode=1)
        orc.step(40)
        try:
            for v in (6, 7, 9):
                print(f"[gpu] march {sc.name} variant {v}", flush=True)
                assert lib().gcomcot_set_tile_variant_(ip(v)) == 0
                dev = DeviceRun(sc)
                dev.run(40)
                compare_device_oracle(sc, dev, orc, f"{sc.name} variant {v}")
                dev.close()
        finally:
            lib().gcomcot_set_tile_variant_(ip(0))


@pytest.mark.parametrize("clc", [0, 1], ids=["sph-child", "cart-child"])
def test_marched_child_matches_oracle(clc):
    """A nested layer wide and tall enough for middle segments: ghost row and
    column, and the ranges of inner layers."""
    from gcomcot._lib import ip, lib
    from helpers import BEACH
    sc = S.custom(nx=110, ny=84, laygov=0, child=dict(laycord=clc, laygov=1, footprint=(51, 41),
                                                      rel_size=4, rel_time=3, corner=(8, 14)), **BEACH)
    orc = Oracle(sc, 32, pow_mode=1)
    orc.step(25)
    try:
        for v in (6, 7, 8, 9, 10):
            print(f"[gpu] march child {clc} variant {v}", flush=True)
            assert lib().gcomcot_set_tile_variant_(ip(v)) == 0
            dev = DeviceRun(sc)
            dev.run(25)
            compare_device_oracle(sc, dev, orc, f"child {clc} variant {v}")
            dev.close()
    finally:
        lib().gcomcot_set_tile_variant_(ip(0))


@pytest.mark.parametrize("count,nx,ny", [(2, 150, 131), (3, 905, 641), (5, 845, 717)],
                         ids=["one-cell-tiles", "strips-of-8", "strips-of-14"])
def test_batched_nonlinear_layers_by_size(count, nx, ny):
    """The shapes that an untuned batch gives nonlinear layers, by the rows
    they have together; one layer is Cartesian, and a linear one beside them
    takes its two steps in marching strips."""
    from gcomcot.batch import Batch
    from helpers import BEACH
    scs = [S.custom(laycord=k % 2, laygov=1, nx=nx - 7 * k, ny=ny - 5 * k, **BEACH) for k in range(count)]
    scs.append(S.custom(laycord=0, laygov=0, nx=331, ny=150))
    print(f"[gpu] batch of {count} nonlinear layers near {nx}x{ny}", flush=True)
    b = Batch(autotune=False, two_step_shape=6)
    sids = [b.add(sc, 15) for sc in scs]
    b.run(15)
    for sc, sid in zip(scs, sids):
        orc = Oracle(sc, 32, pow_mode=1)
        orc.step(15)
        st, mx, o, om = b.state(sid), b.maxima(sid), orc.state(1), orc.maxima(1)
        for k in ("z1", "m1", "n1"):
            nb, worst = diff_report(st[k], o[k])
            assert nb == 0, f"{sc.name} {k}: {nb} cells differ (max {worst})"
        assert diff_report(mx["zmax_wet"], om["zmax_wet"])[0] == 0, sc.name
        assert (mx["arrival"] == om["arrival"]).all(), sc.name
    b.close()


@pytest.mark.parametrize("gov", [0, 1], ids=["linear", "nonlinear"])
@pytest.mark.parametrize("rs,rt", [(3, 1), (2, 2), (4, 4), (7, 5), (3, 9), (5, 21)],
                         ids=["rt1", "rt2", "rt4", "rt5", "rt9", "rt21"])
def test_substeps_that_share_a_jnq_match_oracle(rs, rt, gov):
    """A nested layer's steps write the boundary fluxes of the sub-step that
    follows, under its wet test: REL_TIMEs on every remainder of what one JNQ
    covers (21 asks for more sub-steps than its table holds), in tiles, in one
    cell per thread, in marching strips and in a batch."""
    from gcomcot._lib import ip, lib
    from gcomcot.batch import Batch
    from helpers import BEACH
    sc = S.custom(nx=70, ny=64, laygov=0, child=dict(laycord=1, laygov=gov, footprint=(31, 27),
                                                     rel_size=rs, rel_time=rt, corner=(8, 14)), **BEACH)
    orc = Oracle(sc, 32, pow_mode=1)
    orc.step(21)
    try:
        for v in (0, 1, 6):
            print(f"[gpu] shared jnq {rs}/{rt} gov {gov} variant {v}", flush=True)
            assert lib().gcomcot_set_tile_variant_(ip(v)) == 0
            dev = DeviceRun(sc)
            dev.run(21)
            compare_device_oracle(sc, dev, orc, f"{rs}/{rt} variant {v}")
            dev.close()
    finally:
        lib().gcomcot_set_tile_variant_(ip(0))
    b = Batch(autotune=False)
    sid = b.add(sc, 21)
    b.run(21)
    for lid in (1, 2):
        st, o = b.state(sid, lid), orc.state(lid)
        for k in ("z1", "m1", "n1"):
            assert diff_report(st[k], o[k])[0] == 0, (lid, k)
    b.close()


@pytest.mark.parametrize("nx,ny", [(24, 22), (61, 23), (62, 40), (63, 29), (64, 31), (124, 33), (126, 25)],
                         ids=lambda v: str(v))
def test_marched_moment_mass_matches_oracle(nx, ny):
    """A nested linear root's momentum with the next step's continuity, at
    sizes around one and two strips (62 columns) and off the segments' rows."""
    sc = S.custom(nx=nx, ny=ny, laygov=0, cx=0.4,
                  child=dict(laycord=1, laygov=0, footprint=(7, 6), rel_size=2, rel_time=2, corner=(6, 8)))
    orc = Oracle(sc, 32, pow_mode=1)
    dev = DeviceRun(sc)
    try:
        for n in (1, 2, 60):
            print(f"[gpu] moment + mass {nx}x{ny} run {n}", flush=True)
            dev.run(n)
            orc.step(n)
            compare_device_oracle(sc, dev, orc, f"moment + mass {nx}x{ny} after {n}")
    finally:
        dev.close()


@pytest.mark.parametrize("clc", [0, 1], ids=["sph-child", "cart-child"])
@pytest.mark.parametrize("nx,ny,foot,rt", [(331, 290, (9, 8), 3), (70, 64, (45, 41), 4), (131, 97, (40, 33), 6)],
                         ids=["wide-root", "wide-child", "even"])
def test_root_beside_child_matches_oracle(nx, ny, foot, rt, clc):
    """The root's momentum + next continuity in one launch with a step of its
    child, where either side has more workgroups than the other (one-cell tiles),
    or one after the other (marching strips); and the JNQ made with its JNZ."""
    from gcomcot._lib import ip, lib
    from helpers import BEACH
    sc = S.custom(nx=nx, ny=ny, laygov=0, child=dict(laycord=clc, laygov=1, footprint=foot, rel_size=3,
                                                     rel_time=rt, corner=(8, 14)), **BEACH)
    orc = Oracle(sc, 32, pow_mode=1)
    orc.step(24)
    try:
        for v in (0, 9):
            print(f"[gpu] root beside child {nx}x{ny} {foot} {clc} variant {v}", flush=True)
            assert lib().gcomcot_set_tile_variant_(ip(v)) == 0
            dev = DeviceRun(sc)
            dev.run(23)
            dev.run(1)
            compare_device_oracle(sc, dev, orc, f"root beside child {nx}x{ny} variant {v}")
            dev.close()
    finally:
        lib().gcomcot_set_tile_variant_(ip(0))


@pytest.mark.parametrize("gov,cord,n,variant", [(1, 0, 9, 0), (1, 1, 300, 0), (1, 0, 24, 9), (1, 1, 1, 2), (0, 0, 257, 0),
                                                (0, 1, 24, 0)],
                         ids=["one-cell-tiles", "many", "strips", "tiles", "linear", "linear-cart"])
def test_gauges_sampled_by_the_next_step(gov, cord, n, variant):
    """A run samples the gauges of a step in the launch of the next one, a run
    of one step in a launch of its own: the same samples, ring wraps included."""
    import numpy as np
    from gcomcot._lib import ip, lib
    from helpers import BEACH
    sc = S.custom(laycord=cord, laygov=gov, nx=150, ny=131, **BEACH)
    x, y = S.layer_coords(sc.layers[0])
    rng = np.random.default_rng(n)
    pts = [(float(rng.uniform(x[0], x[-1])), float(rng.uniform(y[0], y[-1])), 1) for _ in range(n)]
    got = []
    try:
        assert lib().gcomcot_set_tile_variant_(ip(variant)) == 0
        for runs in ([19, 1, 5], [1] * 25):
            print(f"[gpu] gauges gov {gov} cord {cord} n {n} variant {variant} runs {len(runs)}", flush=True)
            dev = DeviceRun(sc)
            dev.set_coords()
            dev.set_gauges(pts, 16)
            for k in runs:
                dev.run(k)
            got.append((dev.gauges(25), dev.state(1)["z1"]))
            dev.close()
    finally:
        lib().gcomcot_set_tile_variant_(ip(0))
    assert np.array_equal(got[0][0].view(np.int32), got[1][0].view(np.int32))
    assert np.array_equal(got[0][1].view(np.int32), got[1][1].view(np.int32))
    assert n == 1 or np.any(got[0][0] != 0)  # a lone gauge may lie where the wave has not come


@pytest.mark.parametrize("cord", [0, 1], ids=["sph", "cart"])
@pytest.mark.parametrize("nx,ny", [(33, 9), (31, 25), (767, 253), (768, 256), (769, 256)], ids=lambda v: str(v))
def test_two_threads_per_cell_matches_oracle(nx, ny, cord):
    """Nonlinear layers either side of 768 tiles of 32x8, the most that take two
    threads per cell, and of a tile or two."""
    from helpers import BEACH
    sc = S.custom(laycord=cord, laygov=1, nx=nx, ny=ny, **BEACH)
    orc = Oracle(sc, 32, pow_mode=1)
    print(f"[gpu] two threads per cell {nx}x{ny} cord {cord}", flush=True)
    dev = DeviceRun(sc)
    dev.run(21)
    orc.step(21)
    compare_device_oracle(sc, dev, orc, f"two threads per cell {nx}x{ny}")
    dev.close()


def test_a_tuned_variant_stays_with_its_layer():
    """What the autotuner picks for one layer is not the next layer's variant."""
    import ctypes
    from gcomcot._lib import ip, lib
    now = lambda: lib().gcomcot_tile_variants_(ctypes.byref(ctypes.c_int(0)), None, None)  # noqa: E731
    assert lib().gcomcot_set_tile_variant_(ip(0)) == 0
    print("[gpu] autotune 905x641", flush=True)
    dev = DeviceRun(S.custom(laycord=0, laygov=1, nx=905, ny=641))
    v, b, _ = dev.autotune(reps=3)
    assert now() == v and b == 0
    dev.close()
    small = DeviceRun(S.custom(laycord=0, laygov=1, nx=64, ny=48))
    assert now() == 0
    small.close()


def test_a_tuned_blocking_stays_with_its_layer():
    """What the autotuner picks for one linear layer is not the next layer's
    temporal blocking mode: the tree's own mode holds there."""
    from gcomcot._lib import ip, lib
    now = lib().gcomcot_temporal_blocking_
    try:
        assert lib().gcomcot_set_temporal_blocking_(ip(5)) == 0
        print("[gpu] autotune linear 1024x768", flush=True)
        dev = DeviceRun(S.custom(laycord=0, laygov=0, nx=1024, ny=768))
        _, b, _ = dev.autotune(reps=3)
        assert now() == b
        dev.close()
        small = DeviceRun(S.custom(laycord=0, laygov=0, nx=64, ny=48))
        assert now() == 5
        _, b, _ = small.autotune(reps=3)
        assert now() == b
        assert lib().gcomcot_set_temporal_blocking_(ip(2)) == 0
        assert now() == 2  # the caller's mode ends the tuned one
        small.close()
    finally:
        lib().gcomcot_set_temporal_blocking_(ip(1))


@pytest.mark.parametrize("gov,cord", [(1, 0), (0, 0), (0, 1)], ids=["nonlinear", "linear", "linear-cart"])
def test_a_tuned_layer_keeps_maxima_in_tiles(gov, cord, tmp_path):
    """A tuned layer that is asked for maximum files, which the marching forms
    cannot keep, runs the tuner's best tile, with the same bits, and its tuned
    form again without them."""
    import ctypes
    import numpy as np
    from gcomcot._lib import ip, lib
    from helpers import BEACH
    variant = lambda: lib().gcomcot_tile_variants_(ctypes.byref(ctypes.c_int(0)), None, None)  # noqa: E731
    mode = lib().gcomcot_temporal_blocking_
    assert lib().gcomcot_set_tile_variant_(ip(0)) == 0
    sc = S.custom(laycord=cord, laygov=gov, nx=905, ny=741, **BEACH)
    print(f"[gpu] tuned layer with maxima gov {gov} cord {cord}", flush=True)
    got = []
    for out_opt in (1, 2):
        dev = DeviceRun(sc)
        v, b, _ = dev.autotune(reps=3)
        assert (variant(), mode()) == (v, b if gov == 0 else 1)
        dev.set_output(tmp_path, iprt=0, out_opt=out_opt)
        if out_opt == 2:
            assert gov == 0 or variant() < 6
        else:
            assert (variant(), mode()) == (v, b if gov == 0 else 1)
        dev.run(14)
        got.append((dev.state(1), dev.maxima(1)))
        dev.close()
    (a, am), (c, cm) = got
    for k in ("z1", "m1", "n1"):
        assert np.array_equal(a[k].view(np.int32), c[k].view(np.int32)), k
    for k in ("zmax_wet", "arrival"):
        assert np.array_equal(am[k].view(np.int32), cm[k].view(np.int32)), k


def test_the_tuner_reports_only_forms_that_its_layer_runs():
    """Variants 6-10 are marching strips: of a layer that cannot take them
    (linear, without friction or convection) the tuner times and reports tiles
    only."""
    cases = [dict(laygov=0, laycord=0), dict(laygov=0, laycord=1), dict(laygov=1, laycord=0, fric_coef=0.0),
             dict(laygov=9, laycord=1)]
    for kw in cases:
        for nx, ny in ((331, 290), (96, 72)):
            print(f"[gpu] tuner's variants {kw} {nx}x{ny}", flush=True)
            dev = DeviceRun(S.custom(nx=nx, ny=ny, **kw))
            v, _, _ = dev.autotune(reps=2)
            dev.close()
            assert v < 6, kw
    child = dict(laycord=1, laygov=0, footprint=(51, 41), rel_size=4, rel_time=3, corner=(8, 14))
    dev = DeviceRun(S.custom(nx=110, ny=84, laygov=0, child=child))
    v, _, _ = dev.autotune(reps=2)
    dev.close()
    assert v < 6


@pytest.mark.parametrize("cord", [0, 1], ids=["sph", "cart"])
@pytest.mark.parametrize("count,nx,ny,shape", [(2, 150, 131, 6), (2, 905, 741, 7), (4, 905, 741, 8)],
                         ids=["one-cell-tiles", "strips-of-8", "strips-of-14"])
def test_batched_nonlinear_layers_of_one_kind_by_size(count, nx, ny, shape, cord):
    """The rule takes the layers of one launch, which are of one coordinate kind,
    together: every layer of the batch is of that kind, and the plan says which
    shape it gave them."""
    from gcomcot.batch import Batch
    from helpers import BEACH
    scs = [S.custom(laycord=cord, laygov=1, nx=nx - 7 * k, ny=ny - 5 * k, **BEACH) for k in range(count)]
    print(f"[gpu] batch of {count} nonlinear layers of kind {cord} near {nx}x{ny}", flush=True)
    b = Batch(autotune=False)
    sids = [b.add(sc, 15) for sc in scs]
    b.run(4)
    shapes = b.plan_shapes()
    assert shapes[shape] > 0 and sum(shapes) == shapes[shape], shapes
    b.run(11)
    for sc, sid in zip(scs, sids):
        orc = Oracle(sc, 32, pow_mode=1)
        orc.step(15)
        st, mx, o, om = b.state(sid), b.maxima(sid), orc.state(1), orc.maxima(1)
        for k in ("z1", "m1", "n1"):
            nb, worst = diff_report(st[k], o[k])
            assert nb == 0, f"{sc.name} {k}: {nb} cells differ (max {worst})"
        assert diff_report(mx["zmax_wet"], om["zmax_wet"])[0] == 0, sc.name
        assert (mx["arrival"] == om["arrival"]).all(), sc.name
    b.close()


@pytest.mark.parametrize("cord", [0, 1], ids=["sph", "cart"])
@pytest.mark.parametrize("count,shape", [(2, 7), (4, 8)], ids=["strips-of-8", "strips-of-14"])
def test_batched_children_in_marching_strips(count, shape, cord):
    """Nested layers of a batch in marching strips, whose sides and ends write
    the boundary fluxes of the sub-step that follows."""
    from gcomcot.batch import Batch
    from helpers import BEACH
    scs = [S.custom(nx=250, ny=210, laygov=0, case=k,
                    child=dict(laycord=cord, laygov=1, footprint=(226 - 2 * k, 185 - k), rel_size=4, rel_time=3,
                               corner=(9, 8)), **BEACH) for k in range(count)]
    print(f"[gpu] batch of {count} nests, children of kind {cord}", flush=True)
    b = Batch(autotune=False, streams=2)  # the nests in one chain
    sids = [b.add(sc, 6) for sc in scs]
    b.run(2)
    shapes = b.plan_shapes()
    assert shapes[shape] > 0 and sum(shapes) == shapes[shape], shapes
    b.run(4)
    for sc, sid in zip(scs, sids):
        orc = Oracle(sc, 32, pow_mode=1)
        orc.step(6)
        for lid in (1, 2):
            st, mx, o, om = b.state(sid, lid), b.maxima(sid, lid), orc.state(lid), orc.maxima(lid)
            for k in ("z1", "m1", "n1"):
                nb, worst = diff_report(st[k], o[k])
                assert nb == 0, f"{sc.name} layer {lid} {k}: {nb} cells differ (max {worst})"
            assert diff_report(mx["zmax_wet"], om["zmax_wet"])[0] == 0, (sc.name, lid)
            assert (mx["arrival"] == om["arrival"]).all(), (sc.name, lid)
    b.close()
