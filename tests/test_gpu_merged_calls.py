"""Each merged call against the single calls it stands for, on the forms those
take beyond the step's: arrays with more levels than the index set, and tiles
inside the domain.  The same bits in every array passed and returned."""
import inspect

import pytest
import torch

pytestmark = pytest.mark.gpu
NY, NX = 43, 75
LEVELS = "c1h c2h c1f c2f c3h c4h c3f c4f fnm fnp fzm fzp rdnw rdn dnw rdzw rdzu znu".split()
PLANES = ("mut mub mu muu muv mudf muave muts msfu msfv msft msfux msfuy msfvx msfvx_inv msfvy msftx msfty mu_tend "
          "mu_ori muave_ori muts_ori mudf_ori").split()
SCALARS = dict(rdx=1e-4, rdy=1.1e-4, dts=13.5, dt=13.5, emdiv=0.01, spec_zone=1, epssm=0.1, t0=300.0, smdiv=0.1, step=2,
               non_hydrostatic=True, top_lid=False, n_moist=7, time_step=60)
PREP = ("calculate_full", "calc_mu_uv", "couple_momentum", "calc_ww_cp", "calc_cq", "calc_alt", "calc_php")


class Case:
    """Index sets and arrays by name, drawn on first use."""

    def __init__(self, nz, kte, tile):
        from pywrf_amd.step import Grid
        g = self.g = Grid(nz, NY, NX)
        g.kde = g.kte = g.kpe = kte
        g.its, g.ite, g.jts, g.jte = g.its + tile[0], g.ite - tile[1], g.jts + tile[2], g.jte - tile[3]
        self.nz, self.kte, self.whole, self.drawn = nz, kte, not any(tile), {}
        self.gen = torch.Generator(device="cuda").manual_seed(nz + kte)

    def plane_set(self, lo, hi):
        """The 24-index set with levels lo .. hi."""
        put = {n: lo for n in (4, 10, 16, 22)} | {n: hi for n in (5, 11, 17, 23)}
        return tuple(put.get(n, v) for n, v in enumerate(self.g.ix24))

    def rnd(self, *shape):
        return torch.rand(*shape, device="cuda", generator=self.gen) - 0.5

    def __getitem__(self, n):
        if n not in self.drawn:
            self.drawn[n] = (
                1.0 + 0.02 * self.rnd(NY, NX) if n in PLANES else 0.5 + 0.1 * self.rnd(self.nz) if n in LEVELS else
                torch.tensor(0.5, device="cuda") if n in ("cf1", "cf2", "cf3") else
                self.rnd(7, self.nz, NY, NX) if n == "moist" else 1.0 + 0.1 * self.rnd(self.nz, NY, NX))
        return self.drawn[n]

    def args(self, name, ix, **more):
        """A call's positional arguments: scalars, arrays by parameter name, the index set."""
        import pywrf_amd
        names = list(inspect.signature(getattr(pywrf_amd.ops(), name)).parameters)
        return (*[more[n] if n in more else SCALARS[n] if n in SCALARS else self[n] for n in names[:-len(ix)]], *ix)


def _copy(a, seen):
    if isinstance(a, torch.Tensor):
        return seen.setdefault(id(a), a.clone())
    return type(a)(_copy(x, seen) for x in a) if isinstance(a, (list, tuple)) else a


def _tensors(a):
    if isinstance(a, torch.Tensor):
        return [a]
    return [t for x in a for t in _tensors(x)] if isinstance(a, (list, tuple)) else []


def _equal(c, args, merged, single, but=()):
    """merged(args) and single(args) on copies of args (aliases kept): equal results, and equal arrays after them
    but for those named in but.  What a call leaves unwritten in a fresh result is NaN."""
    runs = []
    for fn in (merged, single):
        seen = {}
        a = _copy(args, seen)
        poison = [torch.full((c.nz, NY, NX), float("nan"), device="cuda") for _ in range(8)]
        poison += [torch.full((NY, NX), float("nan"), device="cuda") for _ in range(8)]
        torch.cuda.synchronize()
        del poison
        runs.append(_tensors(fn(a)) + [seen[id(t)] for n, t in c.drawn.items() if id(t) in seen and n not in but])
    assert len(runs[0]) == len(runs[1])
    for m, (x, y) in enumerate(zip(*runs)):
        assert x.shape == y.shape and torch.equal(torch.nan_to_num(x, nan=3e38), torch.nan_to_num(y, nan=3e38)), m


FORMS = [(41, 41, (0, 0, 0, 0)), (49, 41, (0, 0, 0, 0)), (60, 33, (0, 0, 0, 0)), (41, 41, (3, 4, 2, 5)),
         (49, 41, (4, 1, 3, 2))]


@pytest.fixture(params=FORMS, ids=str)
def case(request):
    return Case(*request.param)


def test_stage_prep(case):
    import pywrf_amd
    o = pywrf_amd.ops()
    calls = [case.args(n, case.g.ix18) for n in PREP]
    _equal(case, calls, lambda a: o.stage_prep(*a), lambda a: [getattr(o, n)(*x) for n, x in zip(PREP, a)])


def test_advect_uvw_fresh(case):
    import pywrf_amd
    o = pywrf_amd.ops()
    calls = [case.args("advect_" + q, case.g.ix18, tendency=case["tend_" + q]) for q in "uvw"]
    _equal(case, calls, lambda a: o.advect_uvw_fresh(*a),
           lambda a: [f(*x) for f, x in zip((o.advect_u_fresh, o.advect_v_fresh, o.advect_w_fresh), a)])


def test_advance_uv_zone(case):
    import pywrf_amd
    o, ix24 = pywrf_amd.ops(), case.g.ix24

    def single(a):
        u, v = o.advance_uv(*a)
        o.spec_bdyupdate(u, a[1], 13.5, "u", 1, *ix24)
        o.spec_bdyupdate(v, a[3], 13.5, "v", 1, *ix24)
        return u, v
    _equal(case, case.args("advance_uv", case.g.ix18), lambda a: o.advance_uv_zone(a, 13.5, ix24), single)


def test_advance_mu_t_zone(case):
    import pywrf_amd
    o, ix24, ix2 = pywrf_amd.ops(), case.g.ix24, case.plane_set(0, 0)

    def single(a):
        r = o.advance_mu_t(*a)
        o.spec_bdyupdate(r[2], a[27], 13.5, "t", 1, *ix24)
        o.spec_bdyupdate(r[10], a[28], 13.5, "m", 1, *ix2)
        o.spec_bdyupdate(r[8], a[28], 13.5, "m", 1, *ix2)
        return r
    _equal(case, case.args("advance_mu_t", case.g.ix18), lambda a: o.advance_mu_t_zone(a, 13.5, ix24, ix2), single)


@pytest.mark.parametrize("iteration,count", [(1, 4), (2, 4), (2, 2), (1, 1)])
def test_sumflux_zone(case, iteration, count):
    import pywrf_amd
    o = pywrf_amd.ops()
    calls = [case.args("sumflux", case.g.ix18, iteration=iteration, number_of_small_timesteps=count),
             case.args("spec_bdyupdate_ph", case.g.ix24, variable_in="h"),
             case.args("zero_grad_bdy", case.g.ix24, field=case["w"], variable_in="w")]
    _equal(case, calls, lambda a: o.sumflux_zone(*a),
           lambda a: [f(*x) for f, x in zip((o.sumflux, o.spec_bdyupdate_ph, o.zero_grad_bdy), a)])


def test_calc_p_rho_bc(case):
    import pywrf_amd
    o, ix24, ix2d = pywrf_amd.ops(), case.g.ix24, case.g.ix2d

    def single(a):
        pr, mudf = a
        r = o.calc_p_rho(*pr)
        o.set_physical_bc_group([(pr[2], "w", 0), (r[0], "p", 0), (r[1], "p", 0), (pr[9], "t", 1), (pr[8], "t", 1),
                                 (mudf, "t", 1)], ix24, ix2d)
        return r
    # (the single call updates pm1 in place, the merged one returns it in a fresh array)
    _equal(case, (case.args("calc_p_rho", case.g.ix18), case["mudf"]),
           lambda a: o.calc_p_rho_bc(a[0], a[1], "wppttt", ix24, ix2d), single, but=("pm1",))


def test_relax_group(case):
    """The mass-weighted fields need mass_weight's box around the whole domain: on a tile without them."""
    import pywrf_amd
    o, g, c = pywrf_amd.ops(), case.g, case
    one = c.plane_set(0, 1)
    weight = (*g.ix24[:12], g.its - 1, g.ite + 1, g.jts - 1, g.jte + 1, 0, c.kte, max(g.its - 1, g.ids),
              min(g.ite + 1, g.ide - 1), max(g.jts - 1, g.jds), min(g.jte + 1, g.jde - 1), 0, c.kte)
    fcx, gcx = torch.linspace(0.0, 0.1, 5, device="cuda"), torch.linspace(0.0, 0.02, 5, device="cuda")
    dtbc = torch.full((1,), 27.0, device="cuda")

    def bdy(kz):
        return tuple(c.rnd(kz, NY, 5) if m % 4 < 2 else c.rnd(kz, 5, NX) for m in range(8))
    mass = c["mut"] if c.whole else None
    items = [(c["ru"], None, c["u_save"], bdy(c.nz), "u", False), (c["rv"], None, c["v_save"], bdy(c.nz), "v", False),
             (c["ph"], mass, c["ph_save"], bdy(c.nz), "h", False), (c["t"], mass, c["t_save"], bdy(c.nz), "t", False),
             (c["mu"].unsqueeze(0), None, c["mu_tend"].unsqueeze(0), bdy(1), "m", True)]

    def merged(its):
        o.relax_group(its, dtbc, fcx, gcx, g.ix24, one, weight)
        return [t for _, _, t, _, _, _ in its]

    def single(its):
        for f, m, t, b, v, two in its:
            if m is not None:
                f = o.mass_weight(f, m, torch.zeros_like(f), c["c1h"], c["c2h"], *weight)
            o.relax_bdytend(f, t, *b, v, 5, 1, 5, dtbc, fcx, gcx, *(one if two else g.ix24))
        return [t for _, _, t, _, _, _ in its]
    _equal(case, items, merged, single)
