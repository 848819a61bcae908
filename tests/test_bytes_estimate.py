"""hobak_inst_bytes_estimate (admission control) covers what an instance allocates, from the smallest mesh on, for
every slice height, layout and precision form (host_engine)."""
import pytest

import host_engine
from hobakv1_amd import lib, scenes


@pytest.mark.parametrize("rows,groups", [(8, 1), (16, 2), (32, 2), (64, 4)])
@pytest.mark.parametrize("precision", [lib.PRECISION_FP64, lib.PRECISION_FP32_REFINE])
@pytest.mark.parametrize("agg", [0, 1])
def test_estimate_covers_the_allocations(monkeypatch, rows, groups, precision, agg):
    monkeypatch.setattr(lib, "_lib", host_engine.load())
    e = host_engine.Engine(slice_rows=rows, update_groups=groups, agg=agg)
    for dims in ((1, 1, 1), (2, 1, 1), (3, 3, 3), (4, 4, 4), (6, 5, 4), (10, 10, 10), (17, 9, 23), (30, 31, 29)):
        sc = scenes.lattice_scene(dims, seed=1)
        before = e.ctx.bytes_in_use()
        inst = lib.Instance(e.ctx, sc, precision=precision)
        assert e.ctx.bytes_in_use() - before <= lib.inst_bytes_estimate(sc.nv, sc.nt, precision), dims
        inst.close()
    e.ctx.close()
