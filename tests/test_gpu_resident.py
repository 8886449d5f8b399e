"""One-launch solves (resident.hip) against the solver launches: the same
bits, for cloths of one part and of many, rows narrower and wider than the
registers hold, both precisions, every lane count whose rounding they follow,
and after a launch that gives up."""
import threading

import numpy as np
import pytest

from acousticsim_amd import capi
from acousticsim_amd import workloads as wl
from obj_fixture import hub_config

pytestmark = pytest.mark.gpu


def _grid(rows, cols, precision, scale=1.0):
    c = wl.grid_config(21, stiffness_scale=scale)
    c["subdivision"] = [rows - 1, cols - 1]
    c["cloth_size"] = [0.5, 0.5 * (cols - 1) / (rows - 1)]
    h, w = (x / 2 for x in c["cloth_size"])
    c["constraints"] = {"static_point": [[-w, h], [w, h]]}
    c["precision"] = precision
    return c, wl.jittered_positions(c, 7)


def _delaunay(points, precision):
    c = wl.delaunay_config(points, size=0.5, seed=3, precision=precision)
    return c, wl.jitter(wl.delaunay_rest_positions(c)[0], 7)


def _run(monkeypatch, cloths, steps, resident, **env):
    monkeypatch.setenv("BW_RESIDENT", resident)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    b = capi.ClothBatch([c for c, _ in cloths], [x for _, x in cloths])
    b.step(steps)
    out = [b.get_pos(i) for i in range(b.n)]
    st = [b.stats(i) for i in range(b.n)]
    b.close()
    for k in env:
        monkeypatch.delenv(k)
    return out, st


ONE_LAUNCH, LANES, LAUNCHES = 2, 1, 0  # solve_route


def _same(a, b, route=ONE_LAUNCH):
    """a's results are b's, a having solved by `route` and b by launches"""
    assert [s["solve_route"] for s in a[1]] == [route] * len(a[1])
    assert not any(s["solve_route"] == ONE_LAUNCH for s in b[1])
    for i, (x, y) in enumerate(zip(a[0], b[0])):
        assert np.array_equal(x, y), "cloth %d" % i
    for p, q in zip(a[1], b[1]):
        for k in ("pcg_iterations", "outer_iterations", "rel_residual", "matrix_fp64"):
            assert p[k] == q[k], (k, p, q)


# vertices: one slice; 7 of 8; one more row than a part holds (FP64: 4
# slices); several parts, ragged
@pytest.mark.parametrize("precision", ["mixed", "fp64"])
@pytest.mark.parametrize("rows,cols", [(2, 2), (5, 5), (21, 21), (16, 16), (17, 16), (32, 16),
                                       (27, 19), (33, 70)])
def test_grid_same_bits(monkeypatch, rows, cols, precision):
    cloth = [_grid(rows, cols, precision)]
    monkeypatch.setenv("BW_SPMV_LPR", "1")
    monkeypatch.setenv("BW_SPMV_STAGE", "0")
    monkeypatch.setenv("BW_SPMV_NT", "0")
    _same(_run(monkeypatch, cloth, 2, "1"), _run(monkeypatch, cloth, 2, "0"))


# clothes whose sums take several rounds of words and of sets: 352 and 1,000
# slices (a round: 1,280 words in FP64, 2,560 in the mixed form; 256 sets)
@pytest.mark.parametrize("rows,cols,precision", [(150, 150, "fp64"), (250, 255, "mixed")])
def test_large_grid_same_bits(monkeypatch, rows, cols, precision):
    cloth = [_grid(rows, cols, precision)]
    monkeypatch.setenv("BW_SPMV_LPR", "1")
    monkeypatch.setenv("BW_SPMV_STAGE", "0")
    monkeypatch.setenv("BW_SPMV_NT", "0")
    _same(*(_run(monkeypatch, cloth, 1, r) for r in "10"))


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
@pytest.mark.parametrize("lpr", ["1", "2", "4"])
def test_lanes_and_wide_rows_same_bits(monkeypatch, lpr, precision):
    """Delaunay rows have up to 25 blocks, 13 of them in registers"""
    cloths = [_delaunay(1200, precision), _grid(40, 40, precision, 5.0), _delaunay(90, precision)]
    monkeypatch.setenv("BW_SPMV_LPR", lpr)
    monkeypatch.setenv("BW_SPMV_STAGE", "0")
    monkeypatch.setenv("BW_SPMV_NT", "0")
    _same(_run(monkeypatch, cloths, 2, "1"), _run(monkeypatch, cloths, 2, "0"))


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
@pytest.mark.parametrize("spokes", [20, 60, 200])
def test_hub_rows_same_bits(monkeypatch, tmp_path, spokes, precision):
    """a vertex with a spoke to each of a ring: its slice alone is wide, its
    blocks past the registers fit in LDS beside the others' (20, 60 in FP32)
    or are read from memory in part"""
    cloth = hub_config(tmp_path / "hub.obj", spokes, precision=precision)
    monkeypatch.setenv("BW_SPMV_LPR", "1")
    monkeypatch.setenv("BW_SPMV_STAGE", "0")
    monkeypatch.setenv("BW_SPMV_NT", "0")
    _same(*(_run(monkeypatch, [cloth], 2, r) for r in "10"))


def test_fp64_matrix_same_bits(monkeypatch):
    """every cloth moved to the FP64 matrix by a check after 20 iterations"""
    cloths = [_grid(40, 33, "mixed", 5.0), _delaunay(700, "mixed")]
    monkeypatch.setenv("BW_SPMV_LPR", "1")
    monkeypatch.setenv("BW_SPMV_STAGE", "0")
    monkeypatch.setenv("BW_SPMV_NT", "0")
    env = dict(BW_MAX_SINCE="20", BW_STALL="1e-9")
    a, b = (_run(monkeypatch, cloths, 2, r, **env) for r in "10")
    assert all(s["matrix_fp64"] for s in a[1])
    _same(a, b, LAUNCHES)  # the second step; the first is in one launch


# one part; several; more slices than launches are faster for; 8 cloths; some
# cloths on the FP32 matrix, so that the others stay beside them
@pytest.mark.parametrize("sides,route", [((21,), ONE_LAUNCH), ((30,), LAUNCHES), ((65, 30), LAUNCHES),
                                         ((97, 97, 97), ONE_LAUNCH), (8 * (30,), ONE_LAUNCH),
                                         ((65, 5), ONE_LAUNCH)])
def test_fp64_matrix_route(monkeypatch, sides, route):
    """steps that start on the FP64 matrix, by the route that is faster there,
    and back after the state is set, with the same bits; a cloth alone leaves
    the launch for that matrix in mid-solve too"""
    cloths = [_grid(n, n, "mixed") for n in sides]
    monkeypatch.setenv("BW_SPMV_LPR", "1")
    # (a 5 x 5 cloth's checks all come within this window)
    monkeypatch.setenv("BW_MAX_SINCE", "20")
    monkeypatch.setenv("BW_STALL", "1e-9")
    out = []
    for resident in "10":
        monkeypatch.setenv("BW_RESIDENT", resident)
        b = capi.ClothBatch([c for c, _ in cloths], [x for _, x in cloths])
        b.step(3)
        st = [b.stats(i) for i in range(b.n)]
        assert [s["matrix_fp64"] for s in st] == [int(n > 5) for n in sides]
        x = [b.get_pos(i) for i in range(b.n)]
        for i in range(b.n):
            b.set_state(i, x[i], x[i])
        b.step(1)
        st += [b.stats(i) for i in range(b.n)]
        out.append(([s["solve_route"] for s in st[:b.n]], [s["solve_route"] for s in st[b.n:]],
                    x, [b.get_pos(i) for i in range(b.n)],
                    [[s[k] for k in ("pcg_iterations", "outer_iterations", "rel_residual")]
                     for s in st]))
        b.close()
    again = LAUNCHES if sides == (30,) else ONE_LAUNCH
    assert out[0][0] == len(sides) * [route] and out[0][1] == len(sides) * [again]
    assert out[0][4] == out[1][4]
    assert not any(r == ONE_LAUNCH for r in out[1][0] + out[1][1])
    for k in (2, 3):
        for p, q in zip(out[0][k], out[1][k]):
            assert np.array_equal(p, q)


def test_more_parts_than_the_chip_holds(monkeypatch):
    """a batch whose parts outnumber the workgroups that run at once"""
    cloths = [_grid(70 + k, 90, "mixed", 0.1) for k in range(28)]
    monkeypatch.setenv("BW_SPMV_LPR", "1")
    monkeypatch.setenv("BW_SPMV_STAGE", "0")
    monkeypatch.setenv("BW_SPMV_NT", "0")
    _same(_run(monkeypatch, cloths, 1, "1"), _run(monkeypatch, cloths, 1, "0"))


@pytest.mark.parametrize("precision,wait_ms", [("mixed", "4"), ("fp64", "8")])
def test_waiting_for_another_cloth_is_no_lost_wait(monkeypatch, precision, wait_ms):
    """waits bounded to less than a solve takes: the parts of a cloth that the
    chip holds only in part wait for the solves before it (with many true
    residuals: the mixed form's progress is seen at every eighth)"""
    monkeypatch.setenv("BW_REL2", "0.5" if precision == "mixed" else "0")
    cloths = [_grid(70 + k, 90, precision, 5.0) for k in range(28)]
    monkeypatch.setenv("BW_SPMV_LPR", "1")
    monkeypatch.setenv("BW_SPMV_STAGE", "0")
    monkeypatch.setenv("BW_SPMV_NT", "0")
    a = _run(monkeypatch, cloths, 1, "1", BW_RESIDENT_WAIT_MS=wait_ms)
    assert max(s["pcg_iterations"] for s in a[1]) > 1500
    _same(a, _run(monkeypatch, cloths, 1, "0"))


def test_batches_of_several_threads_step_side_by_side():
    """a cloth of one part does not wait for another thread's long solves, and
    clothes of several parts, together more than the chip holds, give the
    results that they give alone"""
    def batch(cloth):
        return capi.ClothBatch([cloth[0]], [cloth[1]])
    big = [_grid(129 + 9 * k, 129, "mixed", 5.0) for k in range(3)] + [_grid(200, 200, "mixed")]
    alone = []
    for cloth in big:
        b = batch(cloth)
        b.step(4)
        alone.append(b.get_pos(0))
        b.close()
    batches = [batch(c) for c in big]
    small = batch(_grid(21, 21, "mixed"))
    small.step(1)
    threads = [threading.Thread(target=b.step, args=(4,)) for b in batches]
    for t in threads:
        t.start()
    steps = 0
    while any(t.is_alive() for t in threads):
        small.step(1)
        steps += 1
    for t in threads:
        t.join()
    for b, x in zip(batches, alone):
        assert np.array_equal(b.get_pos(0), x) and b.stats(0)["solve_route"] == ONE_LAUNCH
    assert small.stats(0)["solve_route"] == ONE_LAUNCH
    # 16 solves of some 10 ms and more, and steps of 1 ms beside them
    assert steps > 3 * 16


def test_given_up_launch_solves_by_launches(monkeypatch):
    """a launch that gives up mid-solve (some cloths solved, others not)
    leaves the step to the launches, with their results"""
    cloths = [_grid(9, 9, "mixed", 0.2), _grid(45, 45, "mixed", 5.0), _grid(30, 30, "mixed")]
    monkeypatch.setenv("BW_SPMV_LPR", "1")
    monkeypatch.setenv("BW_SPMV_STAGE", "0")
    monkeypatch.setenv("BW_SPMV_NT", "0")
    _same(_run(monkeypatch, cloths, 2, "1", BW_RESIDENT_GIVE_UP="150"),
          _run(monkeypatch, cloths, 2, "0"), LAUNCHES)


@pytest.mark.parametrize("env", [{}, dict(BW_MAX_SINCE="20", BW_STALL="1e-9")])
def test_given_up_launch_keeps_the_rounding(monkeypatch, env):
    """the steps after a launch that gave up, whose launches are then tuned,
    are those of one-launch solves (no variant fixed by the environment: the
    tuner alone picks 4 lanes for the first two clothes and 2 for the third),
    also of a cloth that stays on the FP64 matrix from step to step"""
    cloths = [_grid(21, 21, "mixed")]
    if not env:
        cloths += [_grid(30, 31, "mixed"), _grid(45, 45, "mixed", 5.0)]
    for cloth in cloths:
        a = _run(monkeypatch, [cloth], 3, "1", BW_RESIDENT_GIVE_UP="150", **env)
        b = _run(monkeypatch, [cloth], 3, "1", **env)
        assert a[1][0]["matrix_fp64"] == b[1][0]["matrix_fp64"] == bool(env)
        assert a[1][0]["solve_route"] == LAUNCHES and b[1][0]["solve_route"] == ONE_LAUNCH
        assert np.array_equal(a[0][0], b[0][0])


def test_lanes_beside_one_launch(monkeypatch):
    """8 clothes whose parts' halos are too long for one launch (their rows
    sorted over the whole mesh) solve in lanes, and the ninth in one launch"""
    monkeypatch.setenv("BW_SORT_WINDOW", "65536")
    monkeypatch.setenv("BW_SPMV_LPR", "1")
    cloths = [_delaunay(7000 + 100 * k, "mixed") for k in range(8)] + [_grid(9, 9, "mixed")]
    a = _run(monkeypatch, cloths, 2, "1")
    b = _run(monkeypatch, cloths, 2, "1", BW_LANES="0")
    assert [s["solve_route"] for s in a[1]] == 8 * [LANES] + [ONE_LAUNCH]
    assert [s["solve_route"] for s in b[1]] == 8 * [LAUNCHES] + [ONE_LAUNCH]
    for x, y in zip(a[0], b[0]):
        assert np.array_equal(x, y)


# the last three: clothes of 11, 17 and 66 parts, from where the parts' sums of
# a true residual, of r.z and r.r, and of d.q reach past the first wavefront's
# words
@pytest.mark.parametrize("rows,cols,max_iters", [(2, 2, 20), (9, 9, 1), (9, 9, 2), (16, 16, 90),
                                                 (17, 16, 90), (33, 70, 150), (52, 53, 150),
                                                 (65, 65, 200), (129, 129, 120)])
def test_reference_semantics_same_bits(monkeypatch, rows, cols, max_iters):
    """the fixed iteration count in one launch against pcg.hip's launches"""
    conf, x0 = _grid(rows, cols, "fp64")
    del conf["precision"]
    conf.update(solver_mode="reference", max_iters=max_iters)
    a, b = (_run(monkeypatch, [(conf, x0), _reference_mesh(max_iters)], 2, r) for r in "10")
    _same(a, b)


def test_reference_semantics_take_no_tuning_window(monkeypatch):
    """BW_MAX_SINCE forces true residuals in the tolerance modes only"""
    conf, x0 = _grid(16, 16, "fp64")
    del conf["precision"]
    conf.update(solver_mode="reference", max_iters=90)
    a = _run(monkeypatch, [(conf, x0)], 2, "1", BW_MAX_SINCE="20")
    _same(a, _run(monkeypatch, [(conf, x0)], 2, "0"))


def _reference_mesh(max_iters):
    conf, x0 = _delaunay(700, "fp64")
    del conf["precision"]
    conf.update(solver_mode="reference", max_iters=max_iters)
    return conf, x0


# pause: iterations after which a round's solves are interrupted; env: a
# cloth on the FP64 matrix, and many true residuals
@pytest.mark.parametrize("precision,pause,env", [
    ("mixed", "", {}), ("mixed", "37", {}), ("fp64", "", {}), ("fp64", "37", {}),
    ("mixed", "1", dict(BW_REL2="0.3")), ("mixed", "13", dict(BW_MAX_SINCE="20", BW_STALL="1e-9"))])
def test_served_same_bits(monkeypatch, precision, pause, env):
    """requests solved together in one launch a round, solves that pause between
    rounds among them, also after a launch that gives up mid-solve, against the
    batch's solver launches"""
    cloths = [_grid(9, 9, precision, 0.2), _delaunay(1200, precision),
              _grid(45, 45, precision, 5.0), _grid(30, 31, precision)]
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    if pause:
        monkeypatch.setenv("BW_RESIDENT_PAUSE", pause)
    monkeypatch.setenv("BW_SPMV_LPR", "1")
    monkeypatch.setenv("BW_SPMV_STAGE", "0")
    monkeypatch.setenv("BW_SPMV_NT", "0")
    ref = _run(monkeypatch, cloths, 2, "0")[0]
    monkeypatch.setenv("BW_RESIDENT", "1")
    # (a launch is given up at a true residual: an FP64 solve's only one ends it)
    for give_up in ("0", "150") if precision == "mixed" else ("0",):
        monkeypatch.setenv("BW_RESIDENT_GIVE_UP", give_up)
        s = capi.Server(budget_bytes=2e9, max_resident=8, precision=precision)
        ids = [s.submit(c, x, 2) for c, x in cloths]
        for rid, x in zip(ids, ref):
            assert s.wait(rid, 60.0) and s.info(rid)["status"] == 0
            assert np.array_equal(s.get_pos(rid), x)
        # a launch a round, or two an iteration of the stiff cloth's hundreds
        iterations = max(s.info(rid)["pcg_iterations"] for rid in ids)
        launches = s.counters()["launches"]
        if give_up != "0":
            assert launches > iterations > 500
        elif pause:
            # (a true residual where a pause is due lets one iteration pass)
            assert iterations // (int(pause) + 1) <= launches < iterations // int(pause) + 100
        else:
            assert launches <= 64
        s.close()


def test_served_by_launches_takes_group_sums(monkeypatch):
    """a served cloth of 520 slices that goes by launches has the sums of those
    above 512 slices, in groups of slices: the bits of a batch with group sums,
    not of one without (in FP64: float vectors round the difference away)"""
    cloth = _grid(182, 182, "fp64", 0.1)
    monkeypatch.setenv("BW_RESIDENT", "0")
    monkeypatch.setenv("BW_SPMV_LPR", "1")
    s = capi.Server(budget_bytes=4e9, max_resident=2, precision="fp64")
    rid = s.submit(cloth[0], cloth[1], 2)
    assert s.wait(rid, 60.0) and s.info(rid)["status"] == 0
    x = s.get_pos(rid)
    s.close()
    monkeypatch.setenv("BW_STAGE_LDS", "p99")
    same = [np.array_equal(x, _run(monkeypatch, [cloth], 2, "0", BW_GROUP_MIN=g)[0][0])
            for g in ("512", "2048")]
    assert same == [True, False]


def test_served_within_a_budget_without_room_for_one_launch(monkeypatch):
    """a budget that holds a request, but not the arrays of its one-launch
    solves, serves it by launches, with the same bits"""
    cloth = _grid(33, 33, "mixed")
    monkeypatch.setenv("BW_SPMV_LPR", "1")

    def serve(budget):
        s = capi.Server(budget_bytes=budget, max_resident=2, precision="mixed")
        rid = s.submit(cloth[0], cloth[1], 2)
        s.wait(rid, 60.0)
        info = s.info(rid)
        x = s.get_pos(rid) if info["status"] == 0 else None
        launches = s.counters()["launches"]
        s.close()
        return info, x, launches
    full, x, few = serve(1e9)
    tight, y, many = serve(full["admitted_bytes"] - 1)
    assert full["status"] == tight["status"] == 0 and np.array_equal(x, y)
    assert few < 100 < tight["pcg_iterations"] < many
    assert tight["device_bytes"] <= tight["admitted_bytes"] < full["admitted_bytes"]
    assert serve(tight["admitted_bytes"] - 1)[0]["status"] == -5  # BW_ERR_CAPACITY


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_served_short_solves_do_not_wait_for_long_ones(precision):
    """20 steps of a 9 x 9 cloth beside a stiff 129 x 129 one whose step takes
    as long: they end within its first steps, not with its 20th"""
    long, x = _grid(129, 129, precision, 10.0)
    short, xs = _grid(9, 9, precision)
    s = capi.Server(budget_bytes=4e9, max_resident=4, precision=precision)
    warm = s.submit(short, xs, 1)
    assert s.wait(warm, 60.0)
    a = s.submit(long, x, 25)
    while s.info(a)["steps_done"] < 1:
        assert not s.wait(a, 0.002)
    b = s.submit(short, xs, 20)
    assert s.wait(b, 60.0) and s.info(b)["status"] == 0
    assert s.info(a)["steps_done"] < 12
    assert s.wait(a, 60.0) and s.info(a)["status"] == 0
    s.close()
