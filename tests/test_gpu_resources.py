"""What a run holds on the device and on the host, what it gives back, and
where its profile keeps its time."""
import ctypes

import pytest
import torch

import chanflow as cf

pytestmark = pytest.mark.gpu


# A run's device memory stays within what cf_run_footprint tells a server's
# budget, but for each of its allocations (30 at most) ending on a 2 MB page:
# rows so short that their spectral partial sums exceed a field, a plane large
# for its levels, the scalar's partial sums of a large grid, the fully implicit
# driver's blocks.
@pytest.mark.parametrize("shape,kw", [((2, 2048, 2000), dict()), ((1024, 1024, 2), dict()), ((512, 512, 400), dict(scalar=1)),
                                      ((256, 256, 97), dict(scalar=1, driver=cf.CF_DRIVER_CHANNEL))])
def test_run_memory_within_footprint(shape, kw):
    cfg = cf.Config(nx=shape[0], ny=shape[1], nz=shape[2], stretch="uniform", **kw)
    cf.Run(cf.Config(nx=16, ny=6, nz=8)).close()          # the library's own memory
    before = torch.cuda.mem_get_info()[0]
    with cf.Run(cfg) as run:
        run.sync()
        used = before - torch.cuda.mem_get_info()[0]
    assert used <= cf.footprint(cfg) + 30 * (2 << 20), (used, cf.footprint(cfg))


# a configuration that is refused after the device was found leaves no live
# run behind: the copies' idle pinned rings go with the last one
def test_refused_run_is_not_counted():
    users = cf.lib().cf_copy_users
    users.argtypes, users.restype = [ctypes.c_int], ctypes.c_int
    live = users(0)
    with pytest.raises(cf.ChanflowError, match="beta"):
        cf.Run(cf.Config(nx=16, ny=6, nz=8, stretch="tanh", stretch_beta=0.0))
    assert users(0) == live
    with cf.Run(cf.Config(nx=16, ny=6, nz=8)):
        assert users(0) == live + 1
    assert users(0) == live


# a solve's time is kept under the name of the solve: nz = 257 has no spike
# tables and takes the Thomas sweep
@pytest.mark.parametrize("nz,solve,other", [(257, "thomas", "spike"), (33, "spike", "thomas")])
def test_solve_time_by_name(nz, solve, other):
    with cf.Run(cf.Config(nx=16, ny=6, nz=nz)) as run:
        run.project(1.0)
        run.set_profiling(True)
        run.step(2)
        run.sync()
        assert run.kernel_time(solve)[1] == 6
        assert run.kernel_time(other)[1] == 0
