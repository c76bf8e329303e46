"""Launch shape of the batched and serving forms: chosen by the content unless the caller gives one."""
import pytest

import mps_gpu as G
from mps_gpu import configs

pytestmark = pytest.mark.gpu


def cube(n, steps):
    m = configs.box(n, n, n)
    dof, val = configs.clamp_bottom_pull_top(m, vel=0.01)
    return dict(mesh=m, dir_dof=dof, dir_val=val, n_steps=steps)


@pytest.mark.parametrize("elem_block,grid_mult", [(0, 0), (128, 4), (64, 0), (0, 3)])
def test_shape_of_the_server(elem_block, grid_mult):
    """A shape that the caller gives is kept and no choice is counted; otherwise 256 work-items per patch and a power of two
    of workgroups per CU."""
    with G.Server(arena_bytes=64 << 20, max_instances=4, elem_block=elem_block, grid_mult=grid_mult) as srv:
        ids = [srv.submit(**cube(n, 64)) for n in (4, 9)]
        assert srv.drain(60.0) == 0
        assert all(srv.result(i)[0] == 0 for i in ids)
        st = srv.stats()
    assert st["elem_block"] == (elem_block or 256)
    assert st["grid_mult"] == grid_mult if grid_mult else st["grid_mult"] in (1, 2, 4, 8, 16)
    assert (st["tunings"] >= 1) == (elem_block == 0 and grid_mult == 0)
