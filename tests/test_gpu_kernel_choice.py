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


# Electrons up and down, walkers, and whether AUTO takes the delayed-update kernel:
# both sides of the lines that its rule has.
LINES = [(4, 4, 8, False), (5, 5, 512, True), (5, 5, 513, False), (6, 6, 1280, True), (6, 6, 1281, False),
         (12, 12, 1281, True), (16, 16, 1281, True), (17, 17, 1280, True), (17, 17, 1281, False),
         (32, 32, 1281, True), (6, 0, 8, False), (8, 0, 512, True), (8, 0, 513, False), (9, 0, 1280, True),
         (14, 0, 1281, True), (17, 0, 1281, False), (24, 0, 1281, True), (8, 1, 8, False), (8, 4, 512, True),
         (8, 4, 513, False), (12, 4, 1280, True), (19, 7, 1281, False), (27, 19, 1281, True)]


@pytest.mark.parametrize("n_up,n_dn,W,delayed", LINES, ids=[f"{a}+{b}_{w}" for a, b, w, _ in LINES])
def test_auto_takes_the_faster_kernel_and_both_follow_one_chain(vmc, n_up, n_dn, W, delayed):
    """The rule's lines; and on either side the chain is that of the other
    kernel: the same number of accepted moves, and positions to the rounding of
    the FP64 proposal (1e-12 L)."""
    s = gas(vmc, n_up, n_dn)
    N, L = s.N, s.box_length
    auto = vmc.Ensemble(s, W, 77 + N, step0=0.5)
    assert auto.kernel() == (vmc.KERNEL_DELAYED if delayed else vmc.KERNEL_GENERIC)
    other = vmc.Ensemble(s, W, 77 + N, step0=0.5)
    other.set_kernel(vmc.KERNEL_GENERIC if delayed else vmc.KERNEL_DELAYED)
    out = []
    for e in (auto, other):
        e.init_positions()
        e.sweep(2, measure=True)
        out.append((e.positions(), e.stats()))
        e.close()
    (p, st), (q, su) = out
    acc, nmeas = vmc.STAT["ACCEPTED"], vmc.STAT["NMEAS"]
    np.testing.assert_array_equal(st[:, acc], su[:, acc])
    assert np.all(st[:, nmeas] == 2) and np.all(su[:, nmeas] == 2)
    np.testing.assert_allclose(p, q, rtol=0, atol=1e-12 * L)


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


def test_a_batch_member_reports_the_kernel_of_its_group(vmc):
    """A batch takes the register kernels or the generic one: an FP64 member
    that alone would take the delayed-update kernel reports the generic one."""
    sy = [gas(vmc, 19, 7), gas(vmc, 27, 27), gas(vmc, 93, 93)]
    b = vmc.Batch(sy, [4, 4, 2], [1, 2, 3])
    fam, grp = b.groups()
    want = [vmc.KERNEL_REGISTER if fam[g] else vmc.KERNEL_GENERIC for g in grp]
    assert [b.member(i).kernel() for i in range(3)] == want
    assert want == [vmc.KERNEL_GENERIC, vmc.KERNEL_REGISTER, vmc.KERNEL_GENERIC]
    b.close()
    for s, k in zip(sy, (vmc.KERNEL_DELAYED, vmc.KERNEL_REGISTER, vmc.KERNEL_DELAYED)):
        e = vmc.Ensemble(s, 4, 1)
        assert e.kernel() == k
        e.close()
