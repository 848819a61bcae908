"""Contexts on two devices used in turn by one thread: every entry point launches on its own context's device
(host_engine)."""
import numpy as np
import pytest

import host_engine
from hobakv1_amd import lib, scenes


@pytest.mark.parametrize("relabelled", [0, 1])
@pytest.mark.parametrize("cells", [4, 40])
def test_every_launch_is_on_its_contexts_device(monkeypatch, relabelled, cells):
    monkeypatch.setattr(lib, "_lib", host_engine.load())
    lib._lib.fake_reset()
    ctxs = [lib.Context(d, apply_table=False) for d in (0, 1)]
    insts = []
    for ctx in ctxs:
        ctx.set_tuning(row_sort=relabelled)
        insts.append(lib.Instance(ctx, scenes.lattice_scene((cells,) * 3, seed=1)))
    u = np.zeros(insts[0].dofs)
    scheds = [lib.Scheduler(ctx) for ctx in ctxs]
    calls = [lambda k: insts[k].set_state(u, u), lambda k: insts[k].state(), lambda k: insts[k].step(True),
             lambda k: lib.step_batch(ctxs[k], [insts[k]], True), lambda k: insts[k].last_system(),
             lambda k: insts[k].forces_hessian(u), lambda k: insts[k].set_pinned([0, 1]),
             lambda k: (scheds[k].submit(insts[k], 0), scheds[k].tick(), scheds[k].tick())]
    for n, call in enumerate(calls):
        for k in (0, 1, 0):
            lib._lib.fake_clear()
            call(k)
            assert lib._lib.fake_wrong_device() == 0, (n, k)
    for s in scheds:
        s.close()
    for i in insts:
        i.close()
    for ctx in ctxs:
        ctx.close()
