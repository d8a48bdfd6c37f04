"""What a run holds on the device and on the host, what it gives back, and
where its profile keeps its time."""
import ctypes

import pytest

import chanflow as cf

pytestmark = pytest.mark.gpu


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
