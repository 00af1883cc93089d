"""GPU parity of the FP64 delayed-update sweep's blocks (vmc_sweep_du.hip).

A block takes up to 32 movers per determinant, 16 below 17 electrons, and
flushes at most 16 accepted moves in row tiles of 16; sizes below sit at the
edges of blocks, tiles and instantiations, with equal spins, unequal spins
(one determinant per block) and one determinant (above 160 electrons the row
tile is read twice).  The device follows the oracle's Philox twin move for
move: positions equal to the rounding of the FP64 proposal (1e-12 L), and the
local energy after each sweep within 1e-9 of the oracle's, the bound the
delayed-update kernel has at its other sizes.
"""
import numpy as np
import pytest

from helpers import oracle_system

pytestmark = pytest.mark.gpu

SIZES = [(1, 0), (2, 1), (8, 1), (16, 16), (17, 17), (19, 7), (7, 19), (32, 32), (34, 33), (48, 48), (49, 49),
         (64, 64), (65, 65), (96, 96), (97, 97), (128, 0), (129, 129), (160, 160), (161, 0), (161, 161), (177, 5),
         (161, 180)]


@pytest.mark.parametrize("n_up,n_dn", SIZES, ids=[f"{a}+{b}" for a, b in SIZES])
def test_blocks_follow_the_oracle_twin(vmc, oracle, n_up, n_dn):
    N = n_up + n_dn
    L = vmc.box_length_from_rs(2.0, N)
    s = vmc.System(n_up, n_dn, L, 0.25, 0.5, 1.0, 5.0 / L, 25, 0.5 * L, vmc.ERFC_EXACT, vmc.MOVE_GAUSSIAN,
                   vmc.PREC_FP64, 0)
    W, seed, step = 2, 700 + N, 0.8
    ens = vmc.Ensemble(s, W, seed, step0=step)
    ens.set_kernel(vmc.KERNEL_DELAYED)
    assert ens.kernel() == vmc.KERNEL_DELAYED
    ens.init_positions()
    osys = oracle_system(oracle, s)
    walkers = [oracle.Walker(osys, oracle.init_positions(osys, seed, w)[0]) for w in range(W)]
    sweeps = 3 if N < 130 else 1
    total = np.zeros(W)
    for sweep in range(sweeps):
        ens.sweep(1, measure=True, adapt=False)
        st, pos = ens.stats(), ens.positions()
        for w in range(W):
            acc, _, e = walkers[w].sweep(seed, w, sweep, step, move_kind=s.move_kind, adapt=False, measure=True)
            total[w] += acc
            np.testing.assert_allclose(pos[w], walkers[w].positions(), rtol=0, atol=1e-12 * L)
            assert st[w, vmc.STAT["ACCEPTED"]] == total[w]
            assert abs(st[w, vmc.STAT["LAST_E"]] - e) <= 1e-9 * max(abs(e), 1e-3 * N), (w, sweep)
    ens.close()


# A smaller determinant beside the one that chose the instantiation: its rows
# end inside a column tile that the larger one's fill, in each instantiation,
# on either side, down to one electron.
SMALLER = [(33, 8), (8, 33), (57, 19), (19, 57), (64, 31), (81, 57), (57, 81), (97, 33), (129, 1), (147, 123)]


@pytest.mark.parametrize("n_up,n_dn", SMALLER, ids=[f"{a}+{b}" for a, b in SMALLER])
def test_the_smaller_determinants_rows_keep_to_themselves(vmc, oracle, n_up, n_dn):
    """The chain of the blocks above with one determinant much smaller, and
    both inverses afterwards those of the final positions, within 1e-9 of
    their largest element (the bound of a chain of delayed updates)."""
    test_blocks_follow_the_oracle_twin(vmc, oracle, n_up, n_dn)
    N = n_up + n_dn
    L = vmc.box_length_from_rs(2.0, N)
    s = vmc.System(n_up, n_dn, L, 0.25, 0.5, 1.0, 5.0 / L, 25, 0.5 * L, vmc.ERFC_EXACT, vmc.MOVE_GAUSSIAN,
                   vmc.PREC_FP64, 0)
    W = 5
    ens = vmc.Ensemble(s, W, 900 + N, step0=0.8)
    ens.set_kernel(vmc.KERNEL_DELAYED)
    ens.init_positions()
    ens.sweep(2, adapt=False)
    inv, pos = ens.inverse(), ens.positions()
    ens.close()
    osys = oracle_system(oracle, s)
    for w in range(W):
        wk = oracle.Walker(osys, pos[w])
        for d, (at, n) in enumerate(((0, n_up), (n_up * n_up, n_dn))):
            ref = wk.inverse(d)
            got = inv[w, at:at + n * n].reshape(n, n)
            assert np.abs(got - ref).max() <= 1e-9 * np.abs(ref).max(), (w, d)


def test_several_sweeps_in_one_launch_are_those_of_single_launches(vmc):
    """Unmeasured sweeps share a launch: the same chain, bit for bit, as one
    launch per sweep, step adaptation included."""
    L = vmc.box_length_from_rs(3.0, 26)
    s = vmc.System(19, 7, L, 0.25, 0.5, 1.0, 5.0 / L, 25, 0.5 * L, vmc.ERFC_EXACT, vmc.MOVE_GAUSSIAN,
                   vmc.PREC_FP64, 0)
    out = []
    for calls, n in ((1, 5), (5, 1)):
        e = vmc.Ensemble(s, 67, 9, step0=0.7)
        e.set_kernel(vmc.KERNEL_DELAYED)
        e.init_positions()
        for _ in range(calls):
            e.sweep(n, adapt=True)
        out.append((e.positions(), e.stats(), e.steps(), e.inverse()))
        e.close()
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("n_up,n_dn,first", [(10, 10, 0), (10, 10, 5), (19, 7, 0), (19, 7, 6), (65, 65, 4), (161, 0, 0),
                                             (161, 0, 9)],
                         ids=["10+10_0", "10+10_5", "19+7_0", "19+7_6", "65+65_4", "161+0_0", "161+0_9"])
def test_a_move_away_from_a_node_keeps_the_inverse(vmc, oracle, n_up, n_dn, first):
    """Two electrons of one spin 1e-5 L apart, one of which (the first mover or
    one in mid-block) moves away: its ratio R is about 1e5 and the inverse
    shrinks by as much.  One rank-1 update leaves an error of a few R roundings
    of the new inverse (n of them in the sums); a flush that multiplied rows R
    times too large by a rounded 1 - (1 - 1/R) left R^2 of them, 1e-6."""
    N = n_up + n_dn
    L = vmc.box_length_from_rs(2.0, N)
    s = vmc.System(n_up, n_dn, L, 0.25, 0.5, 1.0, 5.0 / L, 25, 0.5 * L, vmc.ERFC_EXACT, vmc.MOVE_GAUSSIAN,
                   vmc.PREC_FP64, 0)
    osys = oracle_system(oracle, s)
    rng = np.random.default_rng(31 * N + first)
    W = 3
    pos = np.stack([oracle.init_positions(osys, 5 + w, w)[0] for w in range(W)])
    pos[:, first] = pos[:, first + 2] + 1e-5 * L * np.array([0.6, -0.5, 0.62])
    pos -= L * np.floor(pos / L)
    prop = pos + rng.normal(0.0, 0.1 * L / N ** (1 / 3), pos.shape)
    prop[:, first] = rng.uniform(0.0, L, (W, 3))
    prop -= L * np.floor(prop / L)
    u = rng.uniform(0.0, 1.0, (W, N))
    u[:, first] = 1e-30
    for kernel in (vmc.KERNEL_DELAYED, vmc.KERNEL_GENERIC):
        e = vmc.Ensemble(s, W, 1)
        e.set_kernel(kernel)
        e.set_positions(pos)
        trace = e.sweep_given(prop, u)
        inv, after = e.inverse(), e.positions()
        e.close()
        assert np.all(trace[:, first, 2] == 1.0)
        seen = 0
        for w in range(W):
            R = np.abs(trace[w, :, 0]).max()
            if R < 1e3:  # (its new place is near a node as well)
                continue
            seen += 1
            ref = oracle.Walker(osys, after[w]).inverse(0)
            got = inv[w, :n_up * n_up].reshape(n_up, n_up)
            err = np.abs(got - ref).max() / np.abs(ref).max()
            print(f"kernel {kernel} R {R:.1e} error {err:.1e}", flush=True)
            assert err <= 16 * n_up * 2.2e-16 * R, (kernel, w)
        assert seen >= 2
