"""The advection adjoints at sizes where a wave's columns, rows and levels run
out (58 columns, two rows, eight levels), and with values the forward never
reads set to NaN: <A(q), lam> = <q, A^T lam> (u and v: A is homogeneous in q,
its upwind choices those of q itself)."""
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


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["scalar", "u", "v", "w"])
@pytest.mark.parametrize("nz,ny,nx", [(9, 24, 24), (41, 27, 69), (17, 69, 136), (40, 131, 126)])
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
