"""The kernels that march up several levels a thread, at plane sizes that give
a thread 1, 3 and 8 levels (41 leaves a remainder of each but the first),
against the oracle's calls: the same floats at every point."""
import pytest
import torch


def _copy(a, device=None, seen=None):
    """Copies of the tensors, one for each distinct one."""
    seen = {} if seen is None else seen
    if isinstance(a, torch.Tensor):
        if id(a) not in seen:
            seen[id(a)] = a.clone() if device is None else a.to(device).clone()
        return seen[id(a)]
    if isinstance(a, (list, tuple)):
        return type(a)([_copy(x, device, seen) for x in a])
    return a


class _First:
    """The step's functions, keeping a copy of the arguments of the first call of some."""

    def __init__(self, ops, names):
        self._ops, self._names, self.args = ops, names, {}

    def __getattr__(self, n):
        f = getattr(self._ops, n)
        if n not in self._names:
            return f

        def rec(*args):
            self.args.setdefault(n, _copy(args))
            return f(*args)
        return rec


def _same(a, b):
    a, b = a.cpu(), b.cpu()
    return a.shape == b.shape and torch.equal(torch.nan_to_num(a, nan=3e38), torch.nan_to_num(b, nan=3e38))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [70, 130, 240])
def test_marching_kernels_equal_the_oracle(n):
    import oracle
    import pywrf_amd
    from pywrf_amd.gen import CONFIGS, synthetic_state
    from pywrf_amd.step import RunConfig, rk3_step
    ops, ro = pywrf_amd.ops(), oracle.ops()
    s = synthetic_state(dict(CONFIGS["config2"], n=n), device="cuda")
    rec = _First(ops, ("advance_uv", "pgf_buoy_coriolis_curvature"))
    rk3_step(s, rec, RunConfig())
    args = rec.args["advance_uv"]
    for got, want in zip(ops.advance_uv(*args), ro.advance_uv(*_copy(args, "cpu"))):
        assert _same(got, want)
    hpg, buoy, cc = rec.args["pgf_buoy_coriolis_curvature"]
    h, b, c = _copy((hpg, buoy, cc), "cpu")
    ops.pgf_buoy_coriolis_curvature(hpg, buoy, cc)
    ru, rv = ro.horizontal_pressure_gradient(*h)
    rw, cqw = ro.pg_buoy_w(*b)
    (r0, r1, r2, u, v, w, _, _, _, mux, muy, mvx, mvy, mtx, mty, f, e, sina, cosa, clat, fnm, fnp, rdx, rdy, *ix) = c
    ru, rv, rw = ro.coriolis(r0, r1, r2, ru, rv, rw, mtx, mty, mux, muy, mvx, mvy, f, e, sina, cosa, fnm, fnp, *ix)
    ru, rv, rw = ro.curvature(r0, r1, r2, u, v, w, ru, rv, rw, mux, muy, mvx, mvy, mtx, mty, clat, fnm, fnp, rdx, rdy,
                              *ix)
    for got, want in zip((hpg[0], hpg[1], buoy[0], buoy[2]), (ru, rv, rw, cqw)):
        assert _same(got, want)
