"""Which form of the PCG a step takes, from the context's counters: the resident PCG over the device, on one
die or on every compute unit where its rules say so, the two-kernel form elsewhere, and no launch that leaves an
instance untouched but where the instance cannot fit.  (The forms agree to the bit, so comparing results does not
show which of them ran.)
"""
import numpy as np
import pytest

from hobakv1_amd import lib, scenes

pytestmark = pytest.mark.gpu

F64, F32 = lib.PRECISION_FP64, lib.PRECISION_FP32_REFINE


def _lattice(dims, seed=3, **kw):
    return scenes.lattice_scene(dims, seed=seed, stretch_velocity=True, **kw)


def _forms(scs, precision, workload="single", resident=512, **tuning):
    with lib.Context(0, precision="fp64" if precision == F64 else "fp32", workload=workload) as ctx:
        ctx.set_tuning(resident=resident, **tuning)
        insts = [lib.Instance(ctx, sc, precision=precision) for sc in scs]
        if len(insts) == 1:
            insts[0].step(True)
        else:
            lib.step_batch(ctx, insts, True)
        for i in insts:
            i.close()
        return ctx.resident_stats()


def _only(stats, form):
    assert stats["aborted"] == 0 and stats[form] > 0, stats
    assert all(stats[f] == 0 for f in ("device", "die", "big") if f != form), stats


@pytest.mark.parametrize("precision", [F64, F32])
@pytest.mark.parametrize("dims,form", [((1, 1, 1), "device"), ((4, 4, 4), "device"), ((10, 10, 10), "die"),
                                       ((17, 9, 23), "die"), ((21, 21, 20), "die"), ((22, 22, 22), "device"),
                                       ((40, 40, 40), "device")])
def test_one_instance(dims, form, precision):
    _only(_forms([_lattice(dims)], precision), form)


@pytest.mark.parametrize("precision", [F64, F32])
def test_batches(precision):
    scs = [_lattice((8, 7, 6 + k), seed=k) for k in range(9)]
    _only(_forms(scs[:8], precision, workload="batch"), "die")
    _only(_forms(scs, precision, workload="batch"), "device")
    many = scenes.batch_instances(count=80, seed=9, lo=3, hi=17)
    stats = _forms(many, precision, workload="batch")
    _only(stats, "device")
    assert stats["device"] >= len(many)


def test_more_rows_than_the_update_workgroups_cover():
    _only(_forms([_lattice((35, 37, 35))], F32, update_wgs=256), "big")
    assert set(_forms([_lattice((35, 37, 35))], F64, update_wgs=256).values()) == {0}


@pytest.mark.parametrize("precision", [F64, F32])
def test_layouts_without_a_resident_form(precision):
    for tuning in (dict(slice_rows=8), dict(update_groups=1), dict(grid_cap=1024), dict(resident=0)):
        assert set(_forms([_lattice((11, 7, 8))], precision, **{"resident": 512, **tuning}).values()) == {0}, tuning


def test_columns_that_do_not_fit():
    """A random numbering couples every workgroup to most of the mesh."""
    sc = _lattice((26, 26, 26))
    perm = np.random.default_rng(1).permutation(sc.nv)
    sc.rest, sc.tets = sc.rest[perm], np.argsort(perm)[sc.tets].astype(np.int32)
    sc.v0 = sc.v0.reshape(-1, 3)[perm].ravel()
    stats = _forms([sc], F64)
    assert stats.pop("aborted") > 0 and set(stats.values()) == {0}
