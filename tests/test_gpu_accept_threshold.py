"""The accept test's exact branch in the register kernels.

Within 1e-5 of the threshold the kernels compare u with R^2 exp(2 dJ) in FP64
(their own exponential) instead of the hardware's FP32 one.  The first move of
each walker is given accept uniforms just below and just above the threshold
that its own recorded ratio and Jastrow change imply: the decision must follow
u to 1e-14 relative (the exponential and the two products are within 8
roundings of 1.1e-16, numpy's exp within one), at two Jastrow strengths.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("strength", [1.0, 12.0], ids=["weak", "strong"])
@pytest.mark.parametrize("n_up,n_dn", [(7, 7), (27, 0), (27, 27), (33, 33)], ids=["7+7", "27", "27+27", "33+33"])
def test_first_move_follows_its_threshold(vmc, n_up, n_dn, strength, prec):
    N, W = n_up + n_dn, 64
    L = vmc.box_length_from_rs(2.0, N)
    mixed = prec == "mixed"
    s = vmc.System(n_up, n_dn, L, 0.25 * strength, 0.5 * strength, 1.0, 5.0 / L, 25, 0.5 * L, 1, vmc.MOVE_GAUSSIAN,
                   vmc.PREC_MIXED if mixed else vmc.PREC_FP64, 64 if mixed else 0)
    rng = np.random.default_rng(100 * n_up + n_dn)
    pos = rng.uniform(0.0, L, (W, N, 3))
    prop = rng.uniform(0.0, L, (W, N, 3))

    def first(u0):
        ens = vmc.Ensemble(s, W, 3, step0=0.5)
        ens.set_kernel(vmc.KERNEL_REGISTER)
        ens.set_positions(pos)
        u = np.full((W, N), 1e300)
        u[:, 0] = u0
        tr = ens.sweep_given(prop, u)
        ens.close()
        return tr[:, 0]

    base = first(1e300)
    R, dj = base[:, 0], base[:, 1]
    threshold = R * R * np.exp(2.0 * dj)
    assert np.all(base[:, 2] == 0.0) and np.all(np.isfinite(threshold))
    inside = np.abs(dj) < 40.0
    for factor, accepted in ((1.0 - 1e-14, 1.0), (1.0 + 1e-14, 0.0), (1.0 - 1e-7, 1.0), (1.0 + 1e-7, 0.0)):
        got = first(threshold * factor)
        assert np.array_equal(got[:, :2], base[:, :2])
        assert np.all(got[inside, 2] == accepted), (factor, np.nonzero(got[inside, 2] != accepted))
