"""initial_dt of a state that another blocking stream is still writing: the
call waits for it, on a handle with its own stream and on the null stream; and
of states on either side of the size up to which the host computes it."""
import ctypes
import re

import numpy as np
import pytest

from apollo_amd import engine as E

from cases import euler_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("null_stream", [False, True])
def test_initial_dt_waits_for_blocking_streams(null_stream):
    torch = pytest.importorskip("torch")
    case = euler_case(n=40, N=3, m=5)
    eng = E.Engine(case.mesh, case.params)
    if null_stream:
        E.lib().apl_set_stream(eng._h, None)
    hip = ctypes.CDLL(re.search(r"/\S*libamdhip64\S*", open("/proc/self/maps").read()).group(0))
    raw = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(raw)) == 0
    before, after = case.state(amp=1e-3), case.state(amp=1e-3, seed=1)
    after[..., 1] += 4.0 * after[..., 0]
    after[..., 4] += 20.0
    q, new = torch.from_numpy(before).cuda(), torch.from_numpy(after).cuda()
    a = torch.randn(2048, 2048, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.ExternalStream(raw.value)):
        for _ in range(20):          # some ms of work before the state is there
            a = a @ a
            a /= a.abs().max()
        q.copy_(new)
    dt = eng.initial_dt(q, 0.5)
    torch.cuda.synchronize()
    assert dt == eng.initial_dt(np.ascontiguousarray(after), 0.5)
    assert dt != eng.initial_dt(before, 0.5)
    eng.close()
    assert hip.hipStreamDestroy(raw) == 0


@pytest.mark.parametrize("m", [4, 5])
@pytest.mark.parametrize("n,N", [(1, 1), (13, 2), (14, 2), (18, 2), (19, 2)])
def test_initial_dt_host_and_device_states(n, N, m):
    """2028 nodes are the last below the limit of 2048 here, 2352 the first above."""
    torch = pytest.importorskip("torch")
    case = euler_case(n=n, N=N, m=m, periodic=False)
    q = case.state(amp=1e-3, seed=n)
    eng = E.Engine(case.mesh, case.params)
    assert eng.initial_dt(torch.from_numpy(q).cuda(), 0.5) == eng.initial_dt(q, 0.5)
    q[0, 1, m - 1] = -1.0                # a negative pressure: NaN speeds are passed over
    assert eng.initial_dt(torch.from_numpy(q).cuda(), 0.5) == eng.initial_dt(q, 0.5)
    eng.close()
