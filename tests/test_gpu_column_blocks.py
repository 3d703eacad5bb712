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
