"""Which PCG form the engine takes after a resident launch left an instance untouched, on the CPU (host_engine)."""
import pytest

import host_engine
from host_engine import LATE, LOST, MISFIT
from hobakv1_amd import lib, scenes

F64, F32 = lib.PRECISION_FP64, lib.PRECISION_FP32_REFINE


@pytest.fixture
def engine(monkeypatch):
    monkeypatch.setattr(lib, "_lib", host_engine.load())
    made = []

    def make(**tuning):
        made.append(host_engine.Engine(**tuning))
        return made[-1]

    yield make
    for e in made:
        e.ctx.close()


def _inst(e, dims, precision=F64, **script):
    inst = lib.Instance(e.ctx, scenes.lattice_scene(dims, seed=1), precision=precision)
    e.script(inst, **script)
    e.log()
    return inst


def _step(e, inst):
    inst.step(True)
    return e.forms()


def test_workgroups_that_did_not_meet_meet_later(engine):
    """40^3: 411 update workgroups; a stall once sends a step to the two-kernel form, for a while and not for good."""
    e = engine()
    inst = _inst(e, (40, 40, 40))
    assert _step(e, inst) == ["device"]
    e.script(inst, device=LATE)
    assert _step(e, inst) == ["device", "spmv"]
    e.script(inst)
    later = [_step(e, inst) for _ in range(200)]
    assert later[0] == ["spmv"] and later[-1] == ["device"]
    assert e.ctx.resident_stats()["late"] == 1


def test_stalls_that_go_on_cost_ever_fewer_waits(engine):
    e = engine()
    inst = _inst(e, (40, 40, 40), device=LATE)
    waits = sum(_step(e, inst)[0] == "device" for _ in range(2000))
    assert 2 <= waits <= 8
    assert e.ctx.resident_stats() == {"device": 0, "die": 0, "big": 0, "aborted": waits, "late": waits,
                                       "lost": 0}


def test_columns_that_do_not_fit_take_more_workgroups_and_then_the_two_kernel_form(engine):
    e = engine()
    inst = _inst(e, (40, 40, 40), device=MISFIT)
    for _ in range(4):
        _step(e, inst)
    assert _step(e, inst) == ["spmv"]
    e.script(inst)
    assert all(_step(e, inst) == ["spmv"] for _ in range(200))


def test_a_die_without_room_leaves_the_device_to_the_instance(engine):
    """Another context's large instance holds most of every die: the step goes on over the device, at once."""
    e = engine()
    inst = _inst(e, (10, 10, 10))
    assert _step(e, inst) == ["die"]
    e.script(inst, die=LATE)
    assert _step(e, inst) == ["die", "device"]
    assert _step(e, inst) == ["device"]
    e.script(inst)
    assert [_step(e, inst) for _ in range(60)][-1] == ["die"]


def test_columns_that_do_not_fit_a_die_keep_only_their_instance_off_it(engine):
    e = engine()
    a, b = _inst(e, (10, 10, 10)), _inst(e, (10, 10, 12), die=MISFIT)
    assert _step(e, b) == ["die", "device"]
    assert _step(e, b) == ["device"]
    assert _step(e, a) == ["die"]


def test_an_instance_on_every_compute_unit_keeps_its_form_through_a_stall(engine):
    """Its sums round differently in the two-kernel form, so that is taken only after several waits in a row."""
    e = engine(update_wgs=256)
    inst = _inst(e, (35, 37, 35), precision=F32, big=LATE)
    e.ctx.set_tuning(max_chunks=1, poll_chunk=2)
    forms = _step(e, inst)
    assert forms[:2] == ["big", "spmv"] and e.ctx.resident_stats()["late"] == 4
    e.script(inst)
    assert [_step(e, inst) for _ in range(200)][-1] == ["big"]


@pytest.mark.parametrize("dims,precision,form", [((10, 10, 10), F64, "die"), ((40, 40, 40), F64, "device"),
                                                 ((10, 10, 10), F32, "die")])
def test_a_solve_whose_workgroups_lost_each_other_starts_again(engine, dims, precision, form):
    e = engine()
    inst = _inst(e, dims, precision=precision, iters=30, sweeps=2 if precision == F32 else 1, **{form: LOST})
    e.ctx.set_tuning(max_chunks=1)
    st = inst.step(True)
    log = [w[0] for w in e.log()]
    assert log.count("begin") == 1  # the step itself began once
    assert st["status"] == 0 and st["total_pcg_iters"] == (60 if precision == F32 else 30)
    assert e.ctx.resident_stats()["lost"] == 1
    e.script(inst, iters=30)
    assert _step(e, inst) == ["device" if form == "die" else "spmv"]
    assert [_step(e, inst) for _ in range(200)][-1] == [form]


def test_a_launch_ends_before_the_wait_of_those_behind_it(engine):
    e = engine(resident=65536)
    inst = _inst(e, (10, 10, 10), iters=5000)
    inst.step(True)
    assert [int(w[3]) for w in e.log() if w[0] == "die"] == [2048] * 3


def _two_kernel_launches(e):
    log = e.log()
    return [w[0] for w in log].count("sample"), [w for w in log if w[0] == "spmv"]


@pytest.mark.parametrize("dims,precision,form", [((10, 10, 10), F64, "die"), ((40, 40, 40), F64, "device"),
                                                 ((35, 37, 35), F32, "big")])
def test_sampling_times_one_launch_and_leaves_the_solve_in_its_form(engine, dims, precision, form):
    """No iterations of the two-kernel form, whose sums may round differently (every compute unit)."""
    e = engine(update_wgs=256 if form == "big" else 512)
    inst = _inst(e, dims, precision=precision, iters=100)
    for every in (1, 2, 64):
        inst.set_kernel_sampling(every)
        inst.step(True)
        sampled, launches = _two_kernel_launches(e)
        assert sampled == 1 and launches == [["spmv", "1"]]
        assert inst.kernel_stats()["spmv_count"] == 1
        inst.set_kernel_sampling(0)


def test_an_instance_that_does_not_fit_is_sampled_as_ever(engine):
    """Its first step tries the resident form, is left untouched and goes on in groups, whose launches are sampled."""
    e = engine(update_wgs=256)
    inst = _inst(e, (35, 37, 35), precision=F32, iters=100, big=MISFIT)
    inst.set_kernel_sampling(1)
    inst.step(True)
    assert inst.kernel_stats()["spmv_count"] > 90


def test_a_batch_of_both_forms_samples_the_whole_batch(engine):
    """A sample is credited with every member's bytes, so it has to be a launch over all of them."""
    e = engine(row_sort=0)
    a, b = _inst(e, (10, 10, 10), iters=100), _inst(e, (26, 26, 26), iters=100, device=MISFIT, die=MISFIT)
    for _ in range(4):
        lib.step_batch(e.ctx, [a, b], True)  # b is in the two-kernel form from here on
    for i in (a, b):
        i.set_kernel_sampling(2)
    e.log()
    lib.step_batch(e.ctx, [a, b], True)
    log = e.log()
    at = [k for k, w in enumerate(log) if w[0] == "sample"]
    assert len(at) == 1 and log[at[0] + 1] == ["spmv", "2"]


def test_a_scheduler_samples_solves_that_start(engine):
    e = engine()
    insts = [_inst(e, (10, 10, 10), iters=40), _inst(e, (10, 10, 12), iters=40)]
    sch = lib.Scheduler(e.ctx)
    sch.set_kernel_sampling(100)
    for k in range(10):
        for i in insts:
            sch.submit(i, k)
    left = 1
    while left:
        _, left = sch.tick()
    sampled, launches = _two_kernel_launches(e)
    assert sampled == 4 and launches == [["spmv", "2"]] * 4  # after 0, 120, 240 and 360 of 400 iterations
    row = [int(i.bsr_pattern()[0][-1]) for i in insts]
    expect = sum(n * 76 + 4 * (i.nv + 1) + 48 * i.nv for n, i in zip(row, insts))
    assert sch.kernel_stats()["spmv_bytes"] == expect
    sch.close()


@pytest.mark.parametrize("compact_pct", [0, 100])
def test_groups_of_the_two_kernel_form_leave_resident_members_out(engine, compact_pct):
    """An instance on every compute unit beside one in the two-kernel form: its sums keep their order."""
    e = engine(update_wgs=256, compact_pct=compact_pct)
    big = _inst(e, (35, 37, 35), precision=F32, iters=100)
    other = _inst(e, (30, 30, 30), precision=F32, iters=100, device=MISFIT)
    for _ in range(4):
        lib.step_batch(e.ctx, [big, other], True)
    e.log()
    lib.step_batch(e.ctx, [big, other], True)
    log = e.log()
    before = log[:[w[0] for w in log].index("big")]  # (afterwards its solve has ended)
    assert ["spmv", "1"] in before and ["spmv", "2"] not in before


def _serve(e, insts, ticks):
    """Ticks of a scheduler whose sessions request their next step as soon as one ends: the launches of each."""
    sch = lib.Scheduler(e.ctx)
    for k, i in enumerate(insts):
        sch.submit(i, k)
    out = []
    for _ in range(ticks):
        for c in sch.tick()[0]:
            sch.submit(insts[c["tag"]], c["tag"])
        out.append(e.log())
    sch.close()
    return out


def test_small_sessions_do_not_wait_for_a_large_one_in_the_two_kernel_form(engine):
    e = engine(slice_rows=64, update_groups=4, agg=0)
    large = _inst(e, (40, 40, 40), precision=F32, iters=1000, device=MISFIT)
    small = [_inst(e, (6, 6, 6 + k), precision=F32, iters=35, sweeps=2) for k in range(4)]
    ticks = _serve(e, [large] + small, 80)
    assert max(sum(w[0] == "spmv" for w in t) for t in ticks[20:]) <= 80  # a step of theirs
