"""Contexts of one process stepping in threads of their own, whose resident launches together need more compute units than
the device has: none of them waits in vain, and each ends bitwise where it ends alone."""
import threading
import time

import numpy as np
import pytest

from hobakv1_amd import lib, scenes

pytestmark = pytest.mark.gpu

F64, F32 = lib.PRECISION_FP64, lib.PRECISION_FP32_REFINE


class _Program:
    def __init__(self, dims, precision, steps, **tuning):
        self.ctx = lib.Context(0, precision="fp64" if precision == F64 else "fp32")
        self.ctx.set_tuning(**tuning)
        self.scene = scenes.lattice_scene(dims, seed=3, stretch_velocity=True)
        self.inst = lib.Instance(self.ctx, self.scene, precision=precision)
        self.steps = steps

    def run(self):
        self.inst.set_state(self.scene.initial_u(), self.scene.initial_v())
        for _ in range(self.steps):
            self.inst.step(True)
        self.end = self.inst.state()

    def close(self):
        self.inst.close()
        self.ctx.close()


@pytest.mark.parametrize("programs", [
    [((35, 37, 35), F32, 30, dict(update_wgs=256)), ((30, 30, 30), F64, 40, {}), ((20, 20, 20), F64, 100, {}),
     ((10, 10, 10), F32, 200, {})],
    [((36, 36, 36), F64, 40, {}), ((36, 36, 35), F64, 40, {}), ((35, 36, 36), F32, 40, {})],
    [((20, 20, 20), F64, 60, {})] * 2 + [((10, 10, 10), F64, 150, {})] * 4])
def test_contexts_in_threads(programs):
    print(f"  {programs}", flush=True)
    ps = [_Program(d, prec, n, **t) for d, prec, n, t in programs]
    for p in ps:
        p.run()
    alone = [p.end for p in ps]
    threads = [threading.Thread(target=p.run) for p in ps]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    stats = [p.ctx.resident_stats() for p in ps]
    for p, (u, v) in zip(ps, alone):
        assert np.array_equal(p.end[0], u) and np.array_equal(p.end[1], v)
    for p in ps:
        p.close()
    assert all(s["late"] == 0 and s["aborted"] == 0 for s in stats), stats


@pytest.mark.parametrize("beside", [((40, 40, 40), F64, {}), ((35, 37, 35), F32, dict(update_wgs=256))])
def test_groups_of_the_two_kernel_form_beside_a_resident_stepper(beside):
    """A mesh beyond the resident form while another thread steps one that fills the device: its launches get compute
    units of their own turns, and a step takes a few times what it takes alone, not as long as the other steps."""
    large = _Program((40, 41, 42), F64, 3, update_wgs=256)
    dims, precision, tuning = beside
    other = _Program(dims, precision, 1, **tuning)
    print(f"  {beside}", flush=True)
    large.run()
    t0 = time.perf_counter()
    large.run()
    alone, end = time.perf_counter() - t0, large.end
    assert large.ctx.resident_stats()["device"] == 0
    other.run()
    stop = threading.Event()

    def step():
        while not stop.is_set():
            other.run()

    thread = threading.Thread(target=step)
    thread.start()
    t0 = time.perf_counter()
    large.run()
    took = time.perf_counter() - t0
    stop.set()
    thread.join()
    assert np.array_equal(large.end[0], end[0]) and np.array_equal(large.end[1], end[1])
    large.close()
    other.close()
    assert took < 5 * alone, (took, alone)
