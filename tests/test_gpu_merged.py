"""The step's merged calls against the single calls they stand for: two steps of
each form from the same state, every array of the state bit for bit, at sizes
whose rows and columns leave partial tiles, with live boundary tendencies."""
from types import SimpleNamespace

import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("n", [24, 37, 70])
def test_merged_step_equals_the_single_calls(n):
    import pywrf_amd
    from pywrf_amd.adjoint import MERGED
    from pywrf_amd.gen import CONFIGS, synthetic_state
    from pywrf_amd.state import clone_state, state_tensors
    from pywrf_amd.step import DeviceClock, RunConfig, rk3_step
    a = synthetic_state(dict(CONFIGS["bdy24"], n=n), device="cuda")
    b = clone_state(a, device="cuda")
    ops = vars(pywrf_amd.ops())
    assert MERGED <= set(ops)
    single = SimpleNamespace(**{k: v for k, v in ops.items() if k not in MERGED})
    clocks = DeviceClock(a), DeviceClock(b)
    for _ in range(2):
        rk3_step(a, pywrf_amd.ops(), RunConfig(), clock=clocks[0])
        rk3_step(b, single, RunConfig(), clock=clocks[1])
    for (name, x), (_, y) in zip(state_tensors(a), state_tensors(b)):
        assert torch.equal(x, y) or bool((torch.isnan(x) == torch.isnan(y)).all() and
                                         torch.equal(torch.nan_to_num(x), torch.nan_to_num(y))), name
