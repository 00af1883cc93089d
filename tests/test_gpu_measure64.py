"""GPU parity of the FP64 local energy from inverses in memory (vmc_measure.hip).

Sizes sit where it begins (below six electrons the generic local energy is
taken) and where its split changes: two, four and eight wavefronts (up to 40,
384 and more electrons), one and several slices of an electron's partners,
electrons in one pass and in two, chunks of 64 electrons whose last one is
short, rows of one to three column steps, unequal spins and one determinant;
reciprocal sums of one and of several tiles of columns and powers (a reach of
1 to 11); and the pair cutoff off, on, and past the range of the fitted erfc.
Kinetic, V_real, V_recip, E_L and J against the FP64 oracle at the same
positions: each within 1e-10 of max(|x|, N x 1 mHa), the bound the FP64
kernels have.
"""
import numpy as np
import pytest

from helpers import oracle_system

pytestmark = pytest.mark.gpu

# n_up, n_dn, alpha L, nmax2, cutoff / L (0: none), erfc
CASES = [(1, 0, 5.0, 25, 0.5, 1), (2, 1, 5.0, 25, 0.5, 1), (3, 2, 5.0, 25, 0.5, 1),
         (3, 3, 5.0, 25, 0.5, 1), (6, 0, 5.0, 25, 0.5, 1), (8, 1, 5.0, 1, 0.5, 1), (17, 23, 5.0, 25, 0.5, 1),
         (21, 20, 5.0, 25, 0.5, 1), (33, 33, 5.0, 25, 0.5, 1), (33, 33, 0.0, 0, 0.0, 0), (34, 31, 8.0, 121, 0.5, 1),
         (64, 64, 5.0, 64, 0.0, 1), (65, 64, 5.0, 49, 0.49, 1), (81, 81, 5.0, 25, 0.5, 1), (150, 0, 5.0, 25, 0.5, 1),
         (147, 147, 5.0, 25, 0.5, 1), (193, 192, 5.0, 9, 0.5, 1)]


@pytest.mark.parametrize("n_up,n_dn,al,nmax2,cut,erfc", CASES, ids=[f"{c[0]}+{c[1]}_nmax{c[3]}" for c in CASES])
def test_parts_match_the_oracle(vmc, oracle, n_up, n_dn, al, nmax2, cut, erfc):
    N = n_up + n_dn
    L = vmc.box_length_from_rs(2.0, N)
    s = vmc.System(n_up, n_dn, L, 0.25, 0.5, 1.0, al / L, nmax2, cut * L, erfc, vmc.MOVE_GAUSSIAN, vmc.PREC_FP64, 0)
    W = 3
    ens = vmc.Ensemble(s, W, 60 + N, step0=0.5)
    ens.init_positions()
    got, pos = ens.measure(), ens.positions()
    ens.close()
    osys = oracle_system(oracle, s)
    for w in range(W):
        wk = oracle.Walker(osys, pos[w])
        e, kin, _ = wk.local_energy()
        ref = dict(KINETIC=kin, VREAL=wk.vreal(), VRECIP=wk.vrecip(), ELOCAL=e, JASTROW=wk.jastrow())
        for k, x in ref.items():
            assert abs(got[k][w] - x) <= 1e-10 * max(abs(x), 1e-3 * N), (w, k, got[k][w], x)


def test_two_electrons_at_one_place(vmc, oracle):
    """A pair at r = 0 (electrons of opposite spin) has 1/r = 1 and no
    derivative, as in the reference."""
    N = 66
    L = vmc.box_length_from_rs(2.0, N)
    s = vmc.System.heg(N, 2.0, 1.0)
    rng = np.random.default_rng(4)
    pos = rng.uniform(0.0, L, (1, N, 3))
    pos[0, 40] = pos[0, 3]
    ens = vmc.Ensemble(s, 1, 5)
    ens.set_positions(pos)
    got = ens.measure()
    ens.close()
    wk = oracle.Walker(oracle_system(oracle, s), pos[0])
    assert abs(got["VREAL"][0] - wk.vreal()) <= 1e-10 * max(abs(wk.vreal()), 1e-3 * N)
    assert abs(got["JASTROW"][0] - wk.jastrow()) <= 1e-10 * max(abs(wk.jastrow()), 1e-3 * N)
    assert np.isfinite(got["KINETIC"][0])


@pytest.mark.parametrize("n_up,n_dn", [(27, 27), (27, 0)], ids=["27+27", "27+0"])
def test_mixed_energy_does_not_depend_on_the_number_of_walkers(vmc, n_up, n_dn):
    """The mixed-precision local energy of 27 per spin takes the Slater rows in
    one trip up to 2048 walkers and in two above: the same walkers give the
    same bits in both, refreshed inverses and statistics included, alone and
    in a batch."""
    N = n_up + n_dn
    L = vmc.box_length_from_rs(2.0, N)
    s = vmc.System(n_up, n_dn, L, 0.25, 0.5, 1.0, 5.0 / L, 25, 0.5 * L, vmc.ERFC_EXACT, vmc.MOVE_GAUSSIAN,
                   vmc.PREC_MIXED, 64)
    out = []
    for W in (2048, 2049):
        e = vmc.Ensemble(s, W, 11, step0=0.4)
        e.init_positions()
        e.sweep(3, measure=True)
        parts = e.measure()
        out.append([a[:2048] for a in (e.positions(), e.inverse(), e.stats(), *parts.values())])
        e.close()
        b = vmc.Batch([s], [W], [11], step0=[0.4])
        b.init_positions()
        b.sweep(3, measure=True)
        m = b.member(0)
        out.append([a[:2048] for a in (m.positions(), m.inverse(), m.stats())])
        b.close()
    for other in out[1:]:
        for x, y in zip(out[0], other):
            np.testing.assert_array_equal(x, y)
