"""The scalar transport with one, two and four rows a wave: a call of several
species against a call for each, which takes one row (compared with the oracle
by the per-call tests), bit for bit, at a size that leaves a remainder of rows,
columns and levels in each."""
import os

import pytest
import torch

NZ, NY, NX, KTE = 41, 234, 244, 39


def _rows(species):
    """Rows a wave at that size, by the dispatch's own rule."""
    import pywrf_amd
    from pywrf_amd.step import Grid
    src = open(os.path.join(os.path.dirname(pywrf_amd.__file__), "csrc", "adv.hip")).read()
    assert "const int R = waves(4, SA_KC) >= 1024L * 8 ? 4 : waves(2, SA_KC) >= 1024L * 4 ? 2 : 1;" in src
    assert "#define SA_OX 58\n" in src and "#define SA_KC 8 " in src
    g = Grid(NZ, NY, NX)
    up = lambda a, b: -(-a // b)

    def waves(rows):
        return up(g.ide - 1 - g.ids, 58) * up(g.jde - 1 - g.jds, rows) * up(KTE - 1, 8) * species
    return 4 if waves(4) >= 8192 else 2 if waves(2) >= 4096 else 1


@pytest.mark.parametrize("species,rows", [(1, 1), (3, 2), (9, 4)])
def test_the_species_take_one_two_and_four_rows(species, rows):
    assert _rows(species) == rows


@pytest.mark.gpu
@pytest.mark.parametrize("species", [3, 9])
def test_several_rows_a_wave_equal_one(species):
    import pywrf_amd
    from pywrf_amd.step import Grid
    g = Grid(NZ, NY, NX)
    g.kde = g.kte = KTE
    gen = torch.Generator(device="cuda").manual_seed(species)
    r = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    field, plane, level = (lambda: r(NZ, NY, NX)), (lambda: 1.0 + 0.1 * r(NY, NX)), (lambda: r(NZ))
    ru, rv, ww, alt, xkmhd = (field() for _ in range(5))
    q = r(species, NZ, NY, NX)
    c1h, c2h, base, fnm, fnp, rdn, rdnw = (level() for _ in range(7))
    mut, mub, mu_old, *msf = (plane() for _ in range(10))

    def run(scs, sce):
        tend, adv = torch.full_like(q, 2.0), torch.full_like(q, float("nan"))
        h, z = torch.full_like(ru, float("nan")), torch.full_like(ru, float("nan"))
        pywrf_amd.ops().rk_scalar_tend(scs, sce, False, 2, 20.0, ru, rv, ww, mut, mub, mu_old, c1h, c2h, alt, q, q, tend,
                                       adv, h, z, field(), base, True, fnm, fnp, *msf, 1e-4, 1.1e-4, rdn, rdnw, 0.0, 0.0,
                                       xkmhd, 0, 0.0, 0, *g.ix18)
        return tend[scs:sce + 1], adv[scs:sce + 1], h, z
    tend, adv, h, z = run(0, species - 1)
    same = lambda a, b: torch.equal(torch.nan_to_num(a, nan=3e38), torch.nan_to_num(b, nan=3e38))
    assert not bool(h.any()) and not bool(z.any())
    for m in range(species):
        t1, a1, _, _ = run(m, m)
        assert same(tend[m], t1[0]) and same(adv[m], a1[0]), m
    assert bool(torch.isfinite(adv[:, :KTE - 1, g.jts:g.jte, g.its:g.ite]).all())
