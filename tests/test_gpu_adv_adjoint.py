"""The advection adjoints at sizes where a wave's 58 columns, a workgroup's four
rows and a march of 3 or of 8 levels run out, and with values the forward never
reads set to NaN: <A(q), lam> = <q, A^T lam> (u and v: A is homogeneous in q,
its upwind choices those of q itself)."""
import os
import re

import pytest
import torch


def _case(nz, ny, nx, seed):
    from pywrf_amd.step import Grid
    gen = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    g = Grid(nz, ny, nx)
    f = {n: r(nz, ny, nx) for n in ("q", "lam", "ru", "rv", "rom")}
    for n in ("ru", "rv", "rom"):            # outside the domain nothing is read
        f[n][:, :g.jds] = f[n][:, g.jde + 1:] = float("nan")
        f[n][:, :, :g.ids] = f[n][:, :, g.ide + 1:] = float("nan")
    for n in ("msfux", "msfuy", "msfvx", "msfvy", "msftx", "msfty"):
        f[n] = 1.0 + 0.05 * torch.rand(ny, nx, generator=gen, device="cuda")
    for n in ("fzm", "fzp", "rdz"):
        f[n] = 0.3 + torch.rand(nz, generator=gen, device="cuda")
    return g, f


def _march(nz, ny, nx):
    """Levels a wave marches at that size, from the dispatch's own line."""
    import pywrf_amd
    from pywrf_amd.step import Grid
    src = open(os.path.join(os.path.dirname(pywrf_amd.__file__), "csrc", "adv_adj.hip")).read()
    line, = re.findall(r"const int kc = \(long\)gx \* \(\(a\.j1 - a\.j0 \+ AA_R - 1\) / AA_R\) \* "
                       r"\(\(g->nz \+ 7\) / 8\) >= (\d+) \? 8 : 3;", src)
    assert re.search(r"#define AA_R 1\b", src)
    g = Grid(nz, ny, nx)
    return 8 if -(-(g.ide - g.ids) // 58) * (g.jde - g.jds) * ((nz + 7) // 8) >= int(line) else 3


SIZES = {(9, 24, 24): 3, (41, 27, 69): 3, (17, 69, 136): 3, (40, 131, 126): 3, (41, 237, 243): 8, (48, 240, 242): 8}


@pytest.mark.parametrize("size", list(SIZES))
def test_the_sizes_take_both_marches(size):
    assert _march(*size) == SIZES[size]


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["scalar", "u", "v", "w"])
@pytest.mark.parametrize("nz,ny,nx", list(SIZES))
def test_transpose(kind, nz, ny, nx):
    from pywrf_amd import adjoint
    g, f = _case(nz, ny, nx, nz + ny + nx)
    q = f["q"].clone().requires_grad_()
    if kind == "scalar":
        y = adjoint.AdvectScalar.apply(q, f["ru"], f["rv"], f["rom"], f["msftx"], f["fzm"], f["fzp"], 0.3, 0.4,
                                       f["rdz"], g.ix18)
    else:
        args = [q, q, q, f["ru"], f["rv"], f["rom"], f["fzm"], f["fzm"], f["msftx"], 60,
                *[f[n] for n in ("msfux", "msfuy", "msfvx", "msfvy", "msftx", "msfty")], f["fzm"], f["fzp"], 0.3, 0.4,
                f["rdz"], *g.ix18]
        y = {"u": adjoint.AdvectU, "v": adjoint.AdvectV, "w": adjoint.AdvectW}[kind].apply(q, args)
    lam = f["lam"].clone()
    lam[:, :g.jds - 1] = float("nan")        # rows the tendency never writes to
    dq, = torch.autograd.grad(y, q, lam)
    assert bool(torch.isfinite(dq).all()) and bool(torch.isfinite(y).all())
    lhs = (y.detach().double()[:, g.jds - 1:] * lam.double()[:, g.jds - 1:]).sum()
    rhs = (q.detach().double() * dq.double()).sum()
    # each product carries a few FP32 roundings of terms of the size of its own factors; the sums are over
    # independent signs, so their difference is below 4 eps times the root of the summed squares times 10
    size = (y.detach().double().square().sum() * lam[:, g.jds - 1:].double().square().sum()).sqrt()
    assert abs(float(lhs - rhs)) <= 4 * 6e-8 * 10 * float(size)
