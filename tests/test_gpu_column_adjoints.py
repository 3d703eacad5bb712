"""The column adjoints (64 columns of a row to a block, the levels dealt out to
its waves) at plane sizes around a block's 63 and 64 columns, against the same
FP64 oracle gradients as at the stock sizes, and with level arrays kept in LDS
and, beyond what it holds, in memory; and the grouped sum."""
from types import SimpleNamespace

import pytest
import torch

import test_gpu_adjoint as stock
from pywrf_amd.gen import CONFIGS


@pytest.mark.gpu
@pytest.mark.parametrize("n", [62, 63, 65])
@pytest.mark.parametrize("which", ["advance_w", "advance_uv", "advance_mu_t"])
def test_column_adjoints_around_a_block(which, n):
    fn = {"advance_w": stock.test_advance_w_adjoint_matches_oracle_autograd,
          "advance_uv": stock.test_advance_uv_adjoint_matches_oracle_autograd,
          "advance_mu_t": stock.test_advance_mu_t_adjoint_matches_oracle_differences}[which]
    fn(dict(CONFIGS["bdy24"], n=n))


@pytest.mark.gpu
@pytest.mark.parametrize("nz", [58, 59, 64])
def test_advance_w_adjoint_is_the_same_from_lds_and_memory(nz):
    """Levels above the model's top (index set unchanged) change nothing at
    and below it, whichever place the level arrays take."""
    import pywrf_amd
    from pywrf_amd import adjoint
    from pywrf_amd.gen import synthetic_state
    from pywrf_amd.step import RunConfig, rk3_step
    s = synthetic_state("bdy24", device="cuda")
    rec = stock._FirstCall(pywrf_amd.ops(), "advance_w")
    rk3_step(s, rec, RunConfig())
    nz0 = s.w.shape[0]

    def padded(a):
        if not isinstance(a, torch.Tensor) or a.dim() not in (1, 3) or a.shape[0] != nz0:
            return a
        out = torch.ones((nz,) + tuple(a.shape[1:]), device=a.device)
        out[:nz0] = a
        return out

    D = adjoint.AdvanceW.DIFF + adjoint.AdvanceW.EXTRA
    from pywrf_amd import wrf_dynamics
    outs = wrf_dynamics.advance_w(*rec.args)
    gen = torch.Generator(device="cuda").manual_seed(5)
    lams = [torch.randn(s.w.shape, device="cuda", generator=gen) for _ in outs]
    grads = []
    for pad in (lambda a: a, padded):             # the forward takes fewer levels: the backward by itself
        ctx = SimpleNamespace(args=[pad(a) for a in rec.args], outs=[pad(o) for o in outs[:2]],
                              needs_input_grad=(True,) * (len(D) + 1))
        grads.append(adjoint.AdvanceW.backward(ctx, *[pad(l) for l in lams]))
    for n, a, b in zip(range(len(D) + 1), *grads):
        assert (a is None and b is None) or torch.equal(a, b[:nz0] if b.dim() == 3 else b), n


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 3, 4, 4099])
def test_sum_group_adds_in_order(n):
    from pywrf_amd.adjoint import _sums
    gen = torch.Generator(device="cuda").manual_seed(n)
    t = [torch.randn(n + 1, device="cuda", generator=gen) for _ in range(6)]
    a, b, c, d = (x[:n].clone() for x in t[:4])
    off = t[4][1:]                                # not 16-byte aligned
    x, y, z = torch.empty_like(a), torch.empty_like(off), t[5][:n].clone()
    want = ((a + b) + c) + d, off + b, z + a       # the last into its own source
    _sums((x, (a, b, c, d)), (y, (off, b)), (z, (z, a)))
    for got, w in zip((x, y, z), want):
        assert torch.equal(got, w)


@pytest.mark.gpu
@pytest.mark.parametrize("nx", [24, 69])
def test_advance_mu_t_adjoint_of_values_the_forward_never_reads(nx):
    """NaN around the columns advance_mu_t updates and above its levels reaches no gradient."""
    import oracle
    from pywrf_amd import adjoint
    from pywrf_amd.step import Grid
    from test_gpu_column_blocks import _args
    nz, ny = 11, 27
    g = Grid(nz, ny, nx)
    args = [a.cuda() if isinstance(a, torch.Tensor) else a
            for a in _args(oracle.ops().advance_mu_t, nz, ny, nx, nx)]
    read = torch.zeros(nz, ny, nx, dtype=torch.bool, device="cuda")
    read[:nz - 1, g.jds:g.jde - 1, g.ids:g.ide - 1] = True     # the box's columns and their neighbours
    gen = torch.Generator(device="cuda").manual_seed(nx)
    D, E = adjoint.AdvanceMuT.DIFF, adjoint.AdvanceMuT.EXTRA
    grads = []
    for fill in (0.0, float("nan")):
        a = list(args)
        for n in (1, 2, 3, 4, 5, 10, 11, 25, 27):              # ww_1, u, u_1, v, v_1, muu, muv, t_1, ft
            a[n] = torch.where(read if a[n].dim() == 3 else read[0], a[n], fill)
        x = [a[n].clone().requires_grad_() for n in D + E]
        out = adjoint.AdvanceMuT.apply(*x[:len(D)], a, *x[len(D):])
        if not grads:
            lams = [torch.randn(o.shape, device="cuda", generator=gen) for o in out]
        grads.append(torch.autograd.grad(out, x, lams))
    for n, p, q in zip(D + E, *grads):
        assert torch.equal(p, q), n
