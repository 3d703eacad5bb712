"""The acoustic column kernels at the level counts and row lengths where a
wave's share of levels changes, against the oracle on the same inputs."""
import inspect

import pytest
import torch

from dual import rel_err

PLANES = "mu_ori mut muave_ori muts_ori muu muv mudf_ori mu_tend mu1 muave muts ht".split()
MASS = "mut muts_ori muu muv muts".split()


def _args(fn, nz, ny, nx, seed):
    """Seeded arguments of an oracle function by parameter name, of the magnitudes the step passes."""
    from pywrf_amd.step import Grid
    gen = torch.Generator().manual_seed(seed)
    rnd = lambda *s: torch.rand(*s, generator=gen) - 0.5
    g = Grid(nz, ny, nx)
    scalars = dict(rdx=1. / 9000., rdy=1. / 9000., dts=13.5, epssm=0.1, t0=300.0, step=2, top_lid=False)
    cf = dict(cf1=torch.tensor(2.0), cf2=torch.tensor(-1.5), cf3=torch.tensor(0.5))
    out = []
    for n in list(inspect.signature(fn).parameters)[:-18]:
        if n in scalars:
            out.append(scalars[n])
        elif n in cf:
            out.append(cf[n])
        elif n.startswith("msf"):
            out.append(1.0 + 0.02 * rnd(ny, nx))
        elif n in MASS:
            out.append(9.0e4 + 1.0e3 * rnd(ny, nx))
        elif n in PLANES:
            out.append(100.0 * rnd(ny, nx))
        elif n in ("dnw", "rdnw", "rdn", "fnm", "fnp", "c1h", "c2h", "c1f", "c2f", "c3h", "c4h", "c3f", "c4f"):
            out.append(0.5 + 0.1 * rnd(nz))
        elif n == "phb":
            out.append(2000.0 * torch.arange(nz).float().view(-1, 1, 1) + 100.0 * rnd(nz, ny, nx))
        elif n in ("c2a", "alt"):
            out.append(1.0 + 0.1 * rnd(nz, ny, nx))
        else:
            out.append(10.0 * rnd(nz, ny, nx) if n not in ("a", "alpha", "gamma") else rnd(nz, ny, nx))
    return out + list(g.ix18)


@pytest.mark.gpu
@pytest.mark.parametrize("name,nz,nx", [("advance_mu_t", nz, nx) for nz, nx in
                                        ((3, 24), (9, 69), (41, 133), (42, 64), (65, 65), (128, 40))] +
                         [("advance_w", nz, nx) for nz, nx in ((4, 24), (9, 69), (32, 65), (41, 133), (42, 64))])
def test_level_and_row_edges(name, nz, nx):
    import oracle
    import pywrf_amd
    fn = getattr(oracle.ops(), name)
    args = _args(fn, nz, 27, nx, 7 * nz + nx)
    dev = [a.cuda() if isinstance(a, torch.Tensor) else a for a in args]
    got = getattr(pywrf_amd.ops(), name)(*dev)
    want = fn(*[a.clone() if isinstance(a, torch.Tensor) else a for a in args])
    # advance_mu_t has no transcendental and one order of operations: the same floats.  advance_w's sinf may
    # differ in its last bit between the libraries: the bound is that of the per-call comparison of a step.
    bound = 0.0 if name == "advance_mu_t" else 1e-4
    for n, (x, y) in enumerate(zip(got, want)):
        assert rel_err(x.cpu(), y) <= bound, (name, n)


def _poison(*tensors):
    """Fill the allocator's free blocks of the tensors' sizes with NaN, so that a point a call leaves
    unwritten in its fresh results does not hold an earlier result."""
    blocks = [torch.full_like(t, float("nan")) for _ in range(4) for t in tensors]
    torch.cuda.synchronize()
    del blocks


def _same(x, y):
    x, y = x.cpu(), y.cpu()
    return torch.equal(torch.nan_to_num(x, nan=3e38), torch.nan_to_num(y, nan=3e38))


@pytest.mark.gpu
@pytest.mark.parametrize("nz,kte", [(49, 41), (60, 41), (73, 65), (80, 60), (128, 17), (128, 66)])
def test_arrays_with_more_levels_than_the_index_set(nz, kte):
    """advance_mu_t copies every level of the columns it does not update, and those above kte of the others:
    its results against the oracle's, and with the zone's updates against the four single calls."""
    import oracle
    import pywrf_amd
    from pywrf_amd.step import Grid
    from pywrf_amd.step import SPEC_ZONE
    ny, nx = 27, 69
    ops, fn = pywrf_amd.ops(), oracle.ops().advance_mu_t
    g = Grid(nz, ny, nx)
    g.kde = g.kte = g.kpe = kte
    args = _args(fn, nz, ny, nx, 7 * nz + kte)[:-18] + list(g.ix18)
    dev = [a.cuda() if isinstance(a, torch.Tensor) else a for a in args]
    want = fn(*[a.clone() if isinstance(a, torch.Tensor) else a for a in args])
    _poison(dev[0], dev[6])
    got = ops.advance_mu_t(*dev)
    for n, (x, y) in enumerate(zip(got, want)):
        assert rel_err(x.cpu(), y) == 0.0, n
    ix2d = tuple(0 if n in (4, 5, 10, 11, 16, 17, 22, 23) else v for n, v in enumerate(g.ix24))
    dt, t, muts, mu = 13.5, got[2], got[8], got[10]
    ft, mu_tend = dev[27], dev[28]
    ops.spec_bdyupdate(t, ft, dt, "t", SPEC_ZONE, *g.ix24)
    ops.spec_bdyupdate(mu, mu_tend, dt, "m", SPEC_ZONE, *ix2d)
    ops.spec_bdyupdate(muts, mu_tend, dt, "m", SPEC_ZONE, *ix2d)
    _poison(dev[0], dev[6])
    zone = ops.advance_mu_t_zone(tuple(dev), dt, g.ix24, ix2d)
    for n, (x, y) in enumerate(zip(zone, got)):
        assert _same(x, y), n
