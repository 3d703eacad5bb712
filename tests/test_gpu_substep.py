"""AcousticSubstep, an acoustic substep and its adjoints as one node: against
the same calls as one autograd Function each, and after a caller has written
into its results."""
import functools

import pytest
import torch

pytestmark = pytest.mark.gpu


@functools.lru_cache(maxsize=None)
def _loop(config):
    import pywrf_amd
    from pywrf_amd import adjoint
    from pywrf_amd.gen import synthetic_state
    from pywrf_amd.step import RunConfig
    s = synthetic_state(config, device="cuda")
    x0, subs = adjoint.record_acoustic_loop(s, pywrf_amd.ops(), RunConfig(), stage=2)
    return x0 + adjoint.loop_forcing(subs) + adjoint.loop_saved(subs), subs


def _per_call(x, calls, forcing, saved):
    """The substep's calls, one Function each."""
    from pywrf_amd import adjoint as A
    st = dict(zip(A.ACOUSTIC_STATE, x))
    uv, z1, mt, z2, wa, sf, pz, cp, bc = calls
    given = forcing is not None
    fc = dict(zip(A.FORCING, forcing)) if given else {"ru_tend": uv[1], "rv_tend": uv[3], "rw_tend": None,
                                                      "t_tend": mt[27], "ph_tend": None, "mu_tend": mt[28]}
    sv = dict(zip(A.SAVED, saved)) if saved is not None else dict.fromkeys(A.SAVED)
    live = lambda *names: [fc[n] if given else None for n in names]
    u, v = A.AdvanceUV.apply(st["u"], fc["ru_tend"], st["v"], fc["rv_tend"], st["p"], st["ph"], st["al"], st["mu"],
                             st["mudf"], uv)
    u, v = A.SpecBdyUpdateGroup.apply(z1, u, v, *live("ru_tend", "rv_tend"))
    ww, t, t_ave, muave, muts, mudf, mu = A.AdvanceMuT.apply(
        u, v, st["ww"], st["mu"], st["muave"], st["muts"], st["mudf"], st["t"], st["t_ave"], fc["t_tend"],
        fc["mu_tend"], mt, sv["u_save"], sv["v_save"], sv["ww1"], sv["t_save"])
    t, mu, muts = A.SpecBdyUpdateGroup.apply(z2, t, mu, muts, *live("t_tend", "mu_tend", "mu_tend"))
    t_ave, w, ph = A.AdvanceW.apply(st["w"], st["ph"], t, t_ave, u, v, muts, muave, ww, wa, fc["rw_tend"],
                                    fc["ph_tend"], sv["w_save"], sv["t_save"], sv["ph_save"])
    ru_m, rv_m, ww_m = A.SumFlux.apply(u, v, ww, st["ru_m"], st["rv_m"], st["ww_m"], sf, sv["u_save"], sv["v_save"],
                                       sv["ww1"])
    ph = A.SpecBdyUpdatePh.apply(ph, muts, pz[0], *live("ph_tend", "mu_tend"), sv["ph_save"])
    w = A.ZeroGradBdy.apply(w, pz[1])
    al, p, pm1 = A.CalcPRho.apply(st["al"], st["p"], ph, t, st["pm1"], mu, muts, cp, sv["t_save"])
    items, ix24, ix2d = bc
    ph, al, p, muts, mu, mudf = A.OpenBoundaryFill.apply([(k, two) for _, k, two in items], ix24, ix2d, ph, al, p,
                                                         muts, mu, mudf)
    new = {"u": u, "v": v, "p": p, "ph": ph, "al": al, "mu": mu, "mudf": mudf, "ww": ww, "muave": muave,
           "muts": muts, "t": t, "t_ave": t_ave, "w": w, "pm1": pm1, "ru_m": ru_m, "rv_m": rv_m, "ww_m": ww_m}
    return [new[n] for n in A.ACOUSTIC_STATE]


def _gradients(fn, inputs, calls, parts, lams, after=None):
    from pywrf_amd import adjoint as A
    x = [f.clone().requires_grad_() for f in inputs]
    n, m = len(A.ACOUSTIC_STATE), len(A.ACOUSTIC_STATE) + len(A.FORCING)
    out = fn(x[:n], calls, x[n:m] if "forcing" in parts else None, x[m:] if "saved" in parts else None)
    kept = [o.detach().clone() for o in out]
    if after:
        after(dict(zip(A.ACOUSTIC_STATE, out)))
    return kept, torch.autograd.grad(out, x, lams, allow_unused=True)


def _lams(inputs, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(f.shape, device="cuda", generator=gen) for f in inputs[:17]]


@pytest.mark.parametrize("substep", [0, 1])
@pytest.mark.parametrize("parts", [(), ("forcing",), ("saved",), ("forcing", "saved")])
def test_one_node_equals_a_node_per_call(parts, substep):
    from pywrf_amd import adjoint as A
    inputs, subs = _loop("bdy24")
    lams = _lams(inputs, 3)
    out, grads = _gradients(A.acoustic_substep, inputs, subs[substep], parts, lams)
    want, ref = _gradients(_per_call, inputs, subs[substep], parts, lams)
    for n, a, b in zip(A.ACOUSTIC_STATE, out, want):
        assert torch.equal(torch.nan_to_num(a), torch.nan_to_num(b)), n
    for n, a, b in zip(A.ACOUSTIC_STATE + A.FORCING + A.SAVED, grads, ref):
        assert (a is None) == (b is None), n
        # the same adjoint kernels; a value that several calls read gets at most four shares, summed in another
        # order: a few FP32 roundings of the largest share, which the sum is not below a hundredth of
        if a is not None:
            assert float((a - b).norm()) <= 1e-5 * float(b.norm()), n


@pytest.mark.parametrize("name", ["w", "ph", "mu", "muts"])
def test_a_result_written_into_leaves_the_gradient(name):
    """The values the backward reads are not the caller's: w, ph, mu and muts of the result can be scaled, filled
    or stepped in place, as the copies a node per call returned could."""
    from pywrf_amd import adjoint as A
    inputs, subs = _loop("bdy24")
    lams = _lams(inputs, 5)
    _, ref = _gradients(A.acoustic_substep, inputs, subs[1], ("forcing", "saved"), lams)

    def write(out):
        with torch.no_grad():
            out[name].mul_(1.5).add_(7.0)
    _, got = _gradients(A.acoustic_substep, inputs, subs[1], ("forcing", "saved"), lams, after=write)
    for n, a, b in zip(A.ACOUSTIC_STATE + A.FORCING + A.SAVED, got, ref):
        assert torch.equal(a, b), n
