"""The step takes its merged calls only from an ops whose single calls are the
library's own: a caller's replacement of any of them is called as before."""
from types import SimpleNamespace

import pytest


def test_the_librarys_ops_offer_the_merged_calls():
    import pywrf_amd
    from pywrf_amd.step import offers_merged
    ops = pywrf_amd.ops()
    assert offers_merged(ops)
    assert offers_merged(SimpleNamespace(**vars(ops)))
    assert offers_merged(SimpleNamespace(**dict(vars(ops), microphysics_driver=None)))   # not one of theirs


def _names():
    from pywrf_amd.step import MERGED_CALLS
    return sorted(set(MERGED_CALLS) | {c for calls in MERGED_CALLS.values() for c in calls})


@pytest.mark.parametrize("name", _names())
def test_a_replaced_call_is_called(name):
    import pywrf_amd
    from pywrf_amd.step import offers_merged
    ops = vars(pywrf_amd.ops())
    assert not offers_merged(SimpleNamespace(**dict(ops, **{name: lambda *a: ops[name](*a)})))
    assert not offers_merged(SimpleNamespace(**{k: v for k, v in ops.items() if k != name}))


def test_the_recorders_and_the_oracle_do_not_offer_them():
    import oracle
    import pywrf_amd
    from pywrf_amd.adjoint import _LoopRecorder, _StageRecorder
    from pywrf_amd.step import offers_merged
    assert not offers_merged(_LoopRecorder(pywrf_amd.ops(), 1))
    assert not offers_merged(_StageRecorder(pywrf_amd.ops(), 2))
    assert not offers_merged(oracle.ops())


@pytest.mark.parametrize("name", _names())
def test_a_call_replaced_in_its_module_is_called(name, monkeypatch):
    """ops() takes its functions from the modules: a wrapper put there is the ops' and the module's alike."""
    import functools
    import pywrf_amd
    from pywrf_amd import wrf_boundary, wrf_dynamics
    from pywrf_amd.step import offers_merged
    mod = next(m for m in (wrf_dynamics, wrf_boundary) if hasattr(m, name))
    own = getattr(mod, name)
    monkeypatch.setattr(mod, name, functools.wraps(own)(lambda *a: own(*a)))
    assert getattr(pywrf_amd.ops(), name) is not own
    assert not offers_merged(pywrf_amd.ops())
    monkeypatch.undo()
    assert offers_merged(pywrf_amd.ops())
