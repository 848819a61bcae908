"""The resident PCG (matrices held on chip for a whole launch, HOBAK_TUNE_RESIDENT) against the
two-kernel iteration.

Both form every sum in the same order, so the bar is bitwise equality of positions, velocities,
iteration and sweep counts: for one workgroup and for several, for meshes that end inside a slice, an update
chunk and an SpMV workgroup, for every slice height and update layout, with steps held in registers
only, in LDS too and streamed, and for solves that go on over several launches.
"""
import numpy as np
import pytest

from hobakv1_amd import lib, scenes

pytestmark = pytest.mark.gpu

F64, F32 = lib.PRECISION_FP64, lib.PRECISION_FP32_REFINE


def _steps(scs, precision, resident, workload="single", steps=2, tuning=None, **kw):
    ctx = lib.Context(0, precision="fp64" if precision == F64 else "fp32", workload=workload)
    ctx.set_tuning(resident=resident, **(tuning or {}))
    insts = [lib.Instance(ctx, sc, precision=precision, **kw) for sc in scs]
    stats = []
    for _ in range(steps):
        st = [insts[0].step(True)] if len(insts) == 1 else lib.step_batch(ctx, insts, True)
        stats.append([(s["status"], s["pcg_iters"], s["refine_iters"]) for s in st])
    out = [i.state() for i in insts]
    for i in insts:
        i.close()
    ctx.close()
    return out, stats


def _same(scs, precision, residents=(512,), **kw):
    print(f"  nt {[s.nt for s in scs][:8]} precision {precision} {kw}", flush=True)
    want, ws = _steps(scs, precision, 0, **kw)
    for n in residents:
        got, gs = _steps(scs, precision, n, **kw)
        assert gs == ws, n
        for i, ((u, v), (uw, vw)) in enumerate(zip(got, want)):
            assert np.array_equal(u, uw) and np.array_equal(v, vw), (n, i)


def _lattice(dims, seed=3, **kw):
    return scenes.lattice_scene(dims, seed=seed, stretch_velocity=True, **kw)


@pytest.mark.parametrize("precision", [F64, F32])
@pytest.mark.parametrize("dims", [(1, 1, 1), (4, 4, 4), (6, 5, 4), (10, 10, 10), (3, 30, 5), (17, 9, 23),
                                  (40, 40, 40)])
def test_one_instance(dims, precision):
    _same([_lattice(dims)], precision, residents=(512, 6) if dims == (10, 10, 10) else (512,))


@pytest.mark.parametrize("precision", [F64, F32])
def test_free_and_jacobi(precision):
    """No pinned vertex (the reduced-precision form's coarse correction) and the point preconditioner."""
    _same([_lattice((9, 8, 7), pin=False)], precision, residents=(512, 4))
    _same([_lattice((9, 8, 7))], precision, precond=scenes.PRECOND_JACOBI)
    _same([_lattice((9, 8, 7), pin=False)], precision, precond=scenes.PRECOND_JACOBI, newton_iters=2)


@pytest.mark.parametrize("precision", [F64, F32])
@pytest.mark.parametrize("rows", [8, 16, 32, 64])
def test_slice_heights_and_update_layouts(rows, precision):
    for groups in (1, 2, 4):
        _same([_lattice((11, 7, 8))], precision, residents=(512, 2), steps=1,
              tuning=dict(slice_rows=rows, update_groups=groups, agg=1 if groups != 4 else 2))


@pytest.mark.parametrize("precision", [F64, F32])
def test_batch_past_the_device(precision):
    """More workgroups than compute units: later instances start as earlier ones end."""
    scs = scenes.batch_instances(count=80, seed=9, lo=3, hi=17)
    _same(scs, precision, residents=(512, 32), workload="batch", steps=1)


@pytest.mark.parametrize("precision", [F64, F32])
def test_workgroups_in_whose_rows_no_spmv_workgroup_begins(precision):
    """(16, 5, 4) cells: 510 rows, update workgroups of 168 and SpMV workgroups of 256; such a workgroup still
    takes part in the wait on p.t, so that z is not overwritten before it has read it."""
    scs = [_lattice((16, 5, 4), seed=k) for k in range(24)]
    for pad in (0, 60):  # one update workgroup's rows each, then packed
        _same(scs + [_lattice((24, 24, 20), seed=90 + k) for k in range(pad // 4)], precision, workload="batch",
              steps=2)


def test_serving_layout_streams_past_the_chip():
    """Four row groups and 64-row slices, unpinned, large enough that steps are streamed."""
    scs = [scenes.serving_instance(k, seed=7) for k in range(6)]
    _same(scs, F32, workload="serving", steps=1)


def test_plane_constraints_and_velocity_form():
    _same([scenes.drop_scene((6, 6, 6))], F64, residents=(512, 6), steps=8)
    sc = _lattice((7, 6, 5))
    sc.integrator = scenes.INTEGRATOR_VELOCITY
    _same([sc], F64)


@pytest.mark.parametrize("precision", [F64, F32])
def test_iteration_limit_and_zero_right_hand_side(precision):
    sc = _lattice((8, 8, 8))
    sc.pcg_max_iters = 7
    _same([sc], precision, residents=(512, 4), steps=1)
    rest = scenes.lattice_scene((5, 5, 5), seed=2, g=0.0)
    _same([rest], precision, steps=1)


def test_unconnected_vertices_and_many_columns():
    """Vertices no tet uses have rows without blocks; a random numbering couples every workgroup to most
    of the mesh, beyond what a workgroup can hold, and runs the two-kernel form."""
    sc = _lattice((6, 6, 6))
    far = np.concatenate([sc.rest, sc.rest[:130] + 5.0])
    sc.rest = far
    sc.v0 = np.zeros(3 * far.shape[0])
    sc.mass_scale = 1000.0
    _same([sc], F64, steps=1)
    sc = _lattice((26, 26, 26))
    perm = np.random.default_rng(1).permutation(sc.nv)
    inv = np.argsort(perm)
    sc.rest, sc.tets = sc.rest[perm], inv[sc.tets].astype(np.int32)
    sc.v0 = sc.v0.reshape(-1, 3)[perm].ravel()
    _same([sc], F64, steps=1)


@pytest.mark.parametrize("dims", [(30, 31, 31), (30, 31, 32)])
def test_row_counts_about_the_limit_of_single_slice_words(dims):
    """31,744 and 32,736 rows: 248 and 256 SpMV workgroups of four 32-row slices, either side of the 255 up to
    which a group that straddles two workgroups is published slice by slice."""
    _same([_lattice(dims)], F32, steps=1)


@pytest.mark.parametrize("precision,pin,tuning", [
    (F64, True, {}), (F32, True, {}), (F32, False, {}), (F32, False, dict(slice_rows=16)),
    (F32, True, dict(slice_rows=64, update_groups=4))])
def test_more_rows_than_the_update_workgroups_cover(precision, pin, tuning):
    """256 update workgroups of 168 (or 336) rows and 49,248 (or 91,125) rows: the form on every compute unit, which
    streams what does not fit and publishes one word per workgroup.  Its sums run in another order, so the
    bar is the parity bar, for one launch, for many, and in a batch beside an ordinary instance.  FP64
    solves take the two-kernel form there."""
    dims = (44, 44, 44) if "update_groups" in tuning else (35, 37, 35)
    big, small = _lattice(dims, pin=pin), _lattice((6, 5, 7))
    tuning = dict(update_wgs=256, **tuning)
    want, ws = _steps([big], precision, 0, steps=1, tuning=tuning)
    for n, scs in ((512, [big]), (6, [big]), (512, [small, big])):
        print(f"  nt {big.nt} precision {precision} {tuning} {n} {len(scs)}", flush=True)
        got, gs = _steps(scs, precision, n, steps=1, tuning=tuning)
        x, y = big.rest.ravel() + got[-1][0], big.rest.ravel() + want[0][0]
        assert np.linalg.norm(x - y) <= 1e-9 * np.linalg.norm(y), n
        assert gs[0][-1][0] == ws[0][0][0] and abs(gs[0][-1][1][0] - ws[0][0][1][0]) <= 1, (n, gs, ws)


@pytest.mark.parametrize("precision", [F64, F32])
def test_one_die_and_all_of_them_in_turn(precision):
    """Up to eight instances run on one die each, more of them over the device; the same instances in turn in both,
    with solves that end in one launch and in several, at the row counts about one and two update workgroups'
    rows a workgroup (5,376 and 10,752 rows)."""
    dims = [(6, 5, 4), (16, 16, 17), (17, 17, 15), (21, 21, 20), (21, 21, 21), (3, 30, 5), (8, 8, 8), (9, 8, 7)]
    scs = [_lattice(d, seed=k) for k, d in enumerate(dims)] + [_lattice((5, 5, 5), seed=20 + k) for k in range(3)]

    def run(resident):
        ctx = lib.Context(0, precision="fp64" if precision == F64 else "fp32", workload="batch")
        ctx.set_tuning(resident=resident)
        insts = [lib.Instance(ctx, sc, precision=precision) for sc in scs]
        its = []
        for group in (insts[:1], insts[:8], insts, insts[3:4], insts[4:5], insts[1:8], insts):
            its += [s["pcg_iters"] for s in lib.step_batch(ctx, group, True)]
        out = [i.state() for i in insts]
        for i in insts:
            i.close()
        ctx.close()
        return out, its

    want, wi = run(0)
    for n in (512, 10):
        got, gi = run(n)
        assert gi == wi, n
        for i, ((u, v), (uw, vw)) in enumerate(zip(got, want)):
            assert np.array_equal(u, uw) and np.array_equal(v, vw), (n, i)
