"""GPU parity of the inverses of given positions (vmc_init.hip).

Sizes sit at the edges of its register tiles (2, 4, 8, ... 40 columns a lane:
up to 8, 16, 32, 48, 64, 96, 128 and 160 electrons of a spin), one past each,
columns that do not fill a group of four, unequal spins and one determinant;
161 is the first that the kernel in memory takes, which serves mixed
precision at every size.  With kappa = n |D^-1|_1
(|D| <= 1, so |D|_inf <= n) Gauss-Jordan with partial pivoting is within a
small multiple of n eps kappa of the inverse and of log|det D|: both are held
to 4 n eps kappa against the FP64 oracle, which has such an error itself, plus
for FP32 inverses their rounding, 2^-24 of each element.
"""
import numpy as np
import pytest

from helpers import oracle_system

pytestmark = pytest.mark.gpu

SIZES = [(1, 0), (2, 1), (8, 3), (9, 8), (16, 15), (17, 4), (32, 32), (33, 31), (48, 48), (49, 2), (64, 63), (65, 65),
         (96, 0), (97, 50), (128, 127), (129, 1), (160, 13), (161, 2)]
EPS = np.finfo(np.float64).eps


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("n_up,n_dn", SIZES, ids=[f"{a}+{b}" for a, b in SIZES])
def test_inverse_and_logdet(vmc, oracle, n_up, n_dn, prec):
    N, W = n_up + n_dn, 2
    L = vmc.box_length_from_rs(2.0, N)
    mixed = prec == "mixed"
    s = vmc.System(n_up, n_dn, L, 0.25, 0.5, 1.0, 5.0 / L, 25, 0.5 * L, 1, vmc.MOVE_GAUSSIAN,
                   vmc.PREC_MIXED if mixed else vmc.PREC_FP64, 64 if mixed else 0)
    ens = vmc.Ensemble(s, W, 70 + N, step0=0.5)
    ens.init_positions()
    pos, inv, parts = ens.positions(), ens.inverse(), ens.measure()
    again = vmc.Ensemble(s, W, 1, step0=0.5)
    again.set_positions(pos)
    assert np.array_equal(again.positions(), pos)
    assert np.array_equal(again.inverse(), inv)
    osys = oracle_system(oracle, s)
    for w in range(W):
        wk = oracle.Walker(osys, pos[w])
        assert not wk.singular
        off = 0
        for d, n in enumerate([n_up, n_dn][:1 + (n_dn > 0)]):
            ref = wk.inverse(d)
            got = inv[w, off:off + n * n].reshape(n, n)
            off += n * n
            tol = 4.0 * n * EPS * n * np.abs(ref).sum(axis=0).max()
            assert np.all(np.abs(got - ref) <= tol * np.abs(ref).max() + (2.0 ** -24 * np.abs(ref) if mixed else 0.0))
            assert abs(parts[f"LOGDET{d}"][w] - wk.logdet(d)) <= tol * max(1.0, abs(wk.logdet(d)))
    if n_up > 1:
        bad = pos.copy()
        bad[1, 0] = bad[1, n_up - 1]
        with pytest.raises(vmc.VmcError) as err:
            again.set_positions(bad)
        assert "non-singular" in str(err.value)
    again.close()
    ens.close()
