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


def test_grid_stays_while_the_content_hovers():
    """A large solve of 250 patches beside a small one of 32 needs two workgroups per CU (256 CUs); when the small one has
    ended, one would do, and the grid and its graph stay."""
    with G.Server(arena_bytes=512 << 20, max_instances=4, precision=G.PREC_FP64) as srv:
        ids = [srv.submit(**cube(40, 6400)), srv.submit(**cube(20, 64))]
        assert srv.drain(60.0) == 0
        assert all(srv.result(i)[0] == 0 for i in ids)
        assert srv.stats()["grid_mult"] == 2


def test_grid_comes_down_with_the_content():
    """From 1,331 patches (8 workgroups per CU) to 11: a quarter of the grid would do."""
    with G.Batch(arena_bytes=1 << 30, max_instances=4) as b:
        big, small = (b.add(**cube(n, 1 << 20)) for n in (70, 14))
        b.step(32)
        b.remove(big)
        b.step(32)
        assert b.query(small)["steps"] == 64
    with G.Server(arena_bytes=1 << 30, max_instances=4, precision=G.PREC_FP64) as srv:
        ids = [srv.submit(**cube(70, 64)), srv.submit(**cube(14, 6400))]
        assert srv.drain(60.0) == 0
        assert all(srv.result(i)[0] == 0 for i in ids)
        assert srv.stats()["grid_mult"] == 1
