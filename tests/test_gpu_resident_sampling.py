"""Kernel sampling beside the resident PCG: the launch that is timed ahead of a solve changes nothing the solve reads, to
the bit, and its bytes are the SpMV's algorithmic ones."""
import numpy as np
import pytest

from hobakv1_amd import lib, scenes

pytestmark = pytest.mark.gpu

F64, F32 = lib.PRECISION_FP64, lib.PRECISION_FP32_REFINE


def _lattice(dims, seed=3, **kw):
    return scenes.lattice_scene(dims, seed=seed, stretch_velocity=True, **kw)


def _bytes(inst, s):
    nnzb = int(inst.bsr_pattern()[0][-1])
    return nnzb * (9 * s + 4) + 4 * (inst.nv + 1) + 2 * 3 * s * inst.nv


@pytest.mark.parametrize("dims,precision,pin,tuning", [
    ([(4, 4, 4)], F64, True, {}), ([(10, 10, 10)], F64, True, {}), ([(22, 22, 22)], F64, True, dict(p_form=2)),
    ([(10, 10, 10)], F32, True, {}), ([(9, 8, 7)], F32, False, {}), ([(22, 22, 22)], F32, True, {}),
    ([(35, 37, 35)], F32, True, dict(update_wgs=256)), ([(35, 37, 35)], F32, False, dict(update_wgs=256)),
    ([(8, 7, 6), (9, 8, 7), (17, 9, 23)], F64, True, {}), ([(5 + k, 8, 7) for k in range(12)], F32, True, {}),
    ([(9, 8, 7), (35, 37, 35)], F32, True, dict(update_wgs=256))])
@pytest.mark.parametrize("every", [1, 16, 1000])
def test_results_do_not_depend_on_sampling(dims, precision, pin, tuning, every):
    print(f"  {dims} precision {precision} pin {pin} {tuning} every {every}", flush=True)
    scs = [_lattice(d, seed=k, pin=pin) for k, d in enumerate(dims)]

    def run(every):
        with lib.Context(0, precision="fp64" if precision == F64 else "fp32", workload="batch") as ctx:
            ctx.set_tuning(**tuning)
            insts = [lib.Instance(ctx, sc, precision=precision) for sc in scs]
            for i in insts:
                i.set_kernel_sampling(every)
            its = []
            for _ in range(2):
                its += [s["pcg_iters"] for s in lib.step_batch(ctx, insts, True)]
            out = [i.state() for i in insts]
            ks = insts[0].kernel_stats()
            stats, total = ctx.resident_stats(), sum(_bytes(i, 8 if precision == F64 else 4) for i in insts)
            for i in insts:
                i.close()
        return out, its, ks, stats, total

    want, wi, _, ws, _ = run(0)
    got, gi, ks, gs, total = run(every)
    assert gi == wi and gs == ws and gs["aborted"] == 0
    for (u, v), (uw, vw) in zip(got, want):
        assert np.array_equal(u, uw) and np.array_equal(v, vw)
    assert ks["spmv_count"] == 2 and ks["spmv_avg_ms"] > 0 and ks["spmv_bytes"] == total
