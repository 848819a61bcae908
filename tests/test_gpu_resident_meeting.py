"""Resident launches whose workgroups do not meet in time (HOBAK_TUNE_RESIDENT_JOIN 0: they never do): the instance is
left untouched and solves in another form, with the same results, and goes back to the resident form later.
"""
import numpy as np
import pytest

from hobakv1_amd import lib, scenes

pytestmark = pytest.mark.gpu

F64, F32 = lib.PRECISION_FP64, lib.PRECISION_FP32_REFINE


def _lattice(dims, seed=3, **kw):
    return scenes.lattice_scene(dims, seed=seed, stretch_velocity=True, **kw)


def _run(scs, precision, joins, resident=512, **tuning):
    """The states after one step for each entry of `joins`, and the counters after each."""
    stats = []
    with lib.Context(0, precision="fp64" if precision == F64 else "fp32", workload="batch") as ctx:
        ctx.set_tuning(resident=resident, **tuning)
        insts = [lib.Instance(ctx, sc, precision=precision) for sc in scs]
        for j in joins:
            ctx.set_tuning(resident_join=j)
            lib.step_batch(ctx, insts, True)
            stats.append(ctx.resident_stats())
        out = [i.state() for i in insts]
        for i in insts:
            i.close()
    return out, stats


@pytest.mark.parametrize("precision", [F64, F32])
@pytest.mark.parametrize("dims,form", [([(10, 10, 10)], "die"), ([(22, 22, 22)], "device"),
                                       ([(8, 7, 6), (9, 8, 7), (17, 9, 23)], "die"),
                                       ([(5 + k, 8, 7) for k in range(12)], "device")])
def test_left_untouched_and_taken_up_again(dims, form, precision):
    scs = [_lattice(d, seed=k) for k, d in enumerate(dims)]
    joins = [1, 0] + [1] * 70
    print(f"  {dims} precision {precision}", flush=True)
    want, _ = _run(scs, precision, joins, resident=0)
    got, stats = _run(scs, precision, joins)
    for (u, v), (uw, vw) in zip(got, want):
        assert np.array_equal(u, uw) and np.array_equal(v, vw)
    assert stats[0][form] > 0 and stats[0]["late"] == 0
    # every instance of several workgroups is late, from one die over the device too
    assert stats[1]["late"] >= len(dims) and stats[1]["late"] == stats[1]["aborted"]
    assert stats[1][form] == stats[0][form]
    assert stats[-1]["late"] == stats[1]["late"] and stats[-1][form] > stats[1][form]


def test_every_compute_unit():
    scs = [_lattice((35, 37, 35))]
    want, _ = _run(scs, F32, [1], resident=0, update_wgs=256)
    got, stats = _run(scs, F32, [0], update_wgs=256, max_chunks=1)
    assert stats[0]["late"] >= 4 and stats[0]["big"] == 0
    assert np.linalg.norm(got[0][0] - want[0][0]) <= 1e-9 * np.linalg.norm(scs[0].rest.ravel() + want[0][0])


@pytest.mark.parametrize("precision", [F64, F32])
def test_a_die_that_gets_too_few_workgroups(precision):
    """(With HOBAK_TUNE_RESIDENT_JOIN 0 a launch brings one workgroup too few to each die.)  Nothing of the launch stays behind:
    the next ones on a die, and over the device, run."""
    scs = [_lattice((10, 10, 10)), _lattice((17, 9, 23))]
    joins = [0] + [1] * 70
    want, _ = _run(scs, precision, joins, resident=0)
    got, stats = _run(scs, precision, joins)
    for (u, v), (uw, vw) in zip(got, want):
        assert np.array_equal(u, uw) and np.array_equal(v, vw)
    assert stats[0]["late"] >= 2 and stats[0]["die"] == stats[0]["device"] == 0
    assert stats[-1]["late"] == stats[0]["late"] and stats[-1]["die"] > 0


@pytest.mark.parametrize("dims,precision,tuning,form", [
    ([(4, 4, 4)], F64, {}, "device"), ([(10, 10, 10)], F64, {}, "die"), ([(10, 10, 10)], F32, {}, "die"),
    ([(22, 22, 22)], F64, {}, "device"), ([(22, 22, 22)], F32, {}, "device"),
    ([(8, 7, 6), (9, 8, 7), (17, 9, 23)], F32, {}, "die"), ([(5 + k, 8, 7) for k in range(12)], F64, {}, "device")])
def test_workgroups_that_lose_each_other(dims, precision, tuning, form):
    """(HOBAK_TUNE_RESIDENT_JOIN 2: every launch counts as such.)  The solve starts again, with the same results."""
    scs = [_lattice(d, seed=k) for k, d in enumerate(dims)]
    joins = [1, 2, 2] + [1] * 140
    want, _ = _run(scs, precision, joins, resident=0, **tuning)
    got, stats = _run(scs, precision, joins, **tuning)
    for (u, v), (uw, vw) in zip(got, want):
        assert np.array_equal(u, uw) and np.array_equal(v, vw)
    assert stats[0]["lost"] == 0 and stats[1]["lost"] >= len(dims) and stats[-1]["lost"] == stats[2]["lost"]
    assert stats[-1][form] > stats[2][form] and stats[-1]["aborted"] == 0


def test_workgroups_on_every_compute_unit_that_lose_each_other():
    scs = [_lattice((35, 37, 35))]
    want, _ = _run(scs, F32, [1, 1], resident=0, update_wgs=256)
    got, stats = _run(scs, F32, [2, 1], update_wgs=256)
    assert stats[0]["lost"] == 4 and np.isfinite(got[0][0]).all()
    assert np.linalg.norm(got[0][0] - want[0][0]) <= 1e-9 * np.linalg.norm(scs[0].rest.ravel() + want[0][0])


@pytest.mark.parametrize("precision", [F64, F32])
def test_newton_iterations_and_plane_constraints_after_a_loss(precision):
    sc = _lattice((9, 8, 7))
    sc.newton_iters = 3
    scs = [sc] + ([scenes.drop_scene((6, 6, 6))] if precision == F64 else [])
    for s in scs:
        want, _ = _run([s], precision, [1, 2, 1, 2], resident=0)
        got, stats = _run([s], precision, [1, 2, 1, 2])
        assert np.array_equal(got[0][0], want[0][0]) and np.array_equal(got[0][1], want[0][1])
        assert stats[-1]["lost"] > 0
