"""The sweep kernel an FP64 ensemble takes by itself, the one a caller asks for
by name and the one the autotuner picks are of one set: what get_kernel reports
can be set again, and a tuned ensemble is not slower than an untuned one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def gas(vmc, n_up, n_dn, precision=0):
    L = vmc.box_length_from_rs(2.0, n_up + n_dn)
    return vmc.System(n_up, n_dn, L, 0.25, 0.5, 1.0, 5.0 / L, 25, 0.5 * L, vmc.ERFC_EXACT, vmc.MOVE_GAUSSIAN,
                      precision, 0)


# Unequal spins, sizes above 160 per spin, register sizes, and the smallest.
SIZES = [(1, 0), (2, 1), (7, 7), (19, 7), (33, 27), (50, 50), (57, 19), (161, 161), (177, 5), (485, 0)]


@pytest.mark.parametrize("n_up,n_dn", SIZES, ids=[f"{a}+{b}" for a, b in SIZES])
def test_the_reported_kernel_can_be_set(vmc, n_up, n_dn):
    for precision in (0, 1):
        e = vmc.Ensemble(gas(vmc, n_up, n_dn, precision), 2, 3)
        k = e.kernel()
        e.set_kernel(k)
        assert e.kernel() == k
        if precision == 0:
            e.set_kernel(vmc.KERNEL_DELAYED)
            assert e.kernel() == vmc.KERNEL_DELAYED
        else:
            with pytest.raises(vmc.VmcError):
                e.set_kernel(vmc.KERNEL_DELAYED)
        e.close()


def test_the_delayed_kernel_is_refused_where_it_does_not_fit(vmc):
    e = vmc.Ensemble(gas(vmc, 513, 0), 1, 3)
    assert e.kernel() == vmc.KERNEL_GENERIC
    with pytest.raises(vmc.VmcError):
        e.set_kernel(vmc.KERNEL_DELAYED)
    e.close()


def test_autotune_considers_the_delayed_kernel_for_unequal_spins(vmc):
    """33 + 27 electrons, 64 walkers: the delayed-update kernel takes about a
    third of the generic one's time, so the tuner, which times both, picks it."""
    s = gas(vmc, 33, 27)
    t = vmc.autotune(s, 64, sweeps=4)
    print("tuning", t, flush=True)
    assert t["kernel"] == vmc.KERNEL_DELAYED
    e = vmc.Ensemble(s, 64, 3)
    e.set_kernel(t["kernel"])
    e.init_positions()
    e.sweep(2, measure=True)
    assert np.all(e.stats()[:, vmc.STAT["NMEAS"]] == 2)
    e.close()
