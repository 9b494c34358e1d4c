"""Lattices of few blocks merge and resolve in one workgroup (k_join); with 17 blocks and more the two kernels do. Both
against the oracle: one block, sixteen, the first count past it, partial and padded blocks, tall tiles that keep the two
kernels, both flip rules, and a mixed engine."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n0,n1,tile_rows", [(64, 64, 16), (256, 256, 0), (64, 1024, 16), (1024, 64, 16), (64, 1030, 16), (1088, 64, 16),
                                             (130, 300, 0), (192, 200, 4), (128, 512, 64), (256, 250, 1)])
@pytest.mark.parametrize("T,rule", [(2.0, 0), (2.2691853, 1), (2.6, 0)])
def test_merge_and_flip_match_the_oracle(swmi, oracle, n0, n1, tile_rows, T, rule):
    print(f"join {n0}x{n1} tile_rows {tile_rows} T {T} rule {rule}", flush=True)
    ref = oracle.PerSite(n0, n1, T, seed=n1, spin_seed=2, flip_rule=rule)
    with swmi.Engine(swmi.LatticeConfig(n0, n1, T, seed=n1, spin_seed=2, tile_rows=tile_rows, flip_rule=rule)) as e:
        for k in range(8):
            _, labels = ref.sweep(record=True)
            e.sweep(1)
            if k % 3 == 1:
                np.testing.assert_array_equal(e.labels(), labels, err_msg=f"labels, sweep {k + 1}")
                assert e.energy_magnetization() == oracle.observables(n0, n1, ref.spins)   # the pending flip, not stored
        np.testing.assert_array_equal(e.spins(), ref.spins)
        assert e.error_flags() == 0


def test_lattices_of_a_joined_engine_equal_their_lone_runs(swmi):
    print("join batch", flush=True)
    cfgs = [swmi.LatticeConfig(n0, n1, T, seed=k, flip_rule=k % 2)
            for k, (n0, n1, T) in enumerate([(256, 256, 2.2), (192, 320, 2.0), (128, 130, 2.5), (64, 300, 2.27), (256, 192, 2.8)])]
    with swmi.Engine(cfgs) as e:
        e.set_schedule(1, sweeps=13)
        e.sweep(40)
        got = [e.spins(i) for i in range(len(cfgs))]
    for k, c in enumerate(cfgs):
        with swmi.Engine(c) as alone:
            alone.sweep(13 if k == 1 else 40)
            np.testing.assert_array_equal(alone.spins(), got[k], err_msg=f"lattice {k}")
            assert alone.error_flags() == 0


@pytest.mark.parametrize("n0,n1", [(64, 262144), (262144, 64), (128, 131074)])
@pytest.mark.parametrize("T", [2.0, 2.2691853])
def test_launches_of_4096_blocks_one_or_two_wide(swmi, oracle, n0, n1, T):
    """From 4096 blocks one wave unites both edges of a block in LDS (k_merge_block). A block that is its own right or
    lower neighbour has each slot twice in that table."""
    print(f"block merge {n0}x{n1} T {T}", flush=True)
    ref = oracle.PerSite(n0, n1, T, seed=3)
    with swmi.Engine(swmi.LatticeConfig(n0, n1, T, seed=3)) as e:
        e.sweep(1)
        _, labels = ref.sweep(record=True)
        np.testing.assert_array_equal(e.labels(), labels)
        np.testing.assert_array_equal(e.spins(), ref.spins)
        e.sweep(1)
        ref.sweep()
        np.testing.assert_array_equal(e.spins(), ref.spins)
        assert e.error_flags() == 0


def test_many_small_tiled_lattices_equal_their_lone_runs(swmi):
    """1040 lattices of two by two blocks in one launch of 4177 blocks: every block meets the same neighbour twice. (The
    lattice of 17 blocks keeps the class off k_join.)"""
    print("block merge, 1040 lattices", flush=True)
    cfgs = [swmi.LatticeConfig(128, 128, 1.9 + 0.001 * i, seed=i, tile_rows=16, flip_rule=i % 2) for i in range(1040)]
    cfgs.append(swmi.LatticeConfig(64, 1088, 2.2, seed=3, tile_rows=16))
    with swmi.Engine(cfgs) as e:
        e.sweep(12)
        got = {i: e.spins(i) for i in range(0, 1041, 13)}
        assert all(e.error_flags(i) == 0 for i in got)
    for i, spins in got.items():
        with swmi.Engine(cfgs[i]) as alone:
            alone.sweep(12)
            np.testing.assert_array_equal(alone.spins(), spins, err_msg=f"lattice {i}")


@pytest.mark.parametrize("n0,n1,T,rule", [(1006, 270, 2.392, 1), (130, 300, 2.0, 0), (256, 258, 2.2691853, 1),
                                          (512, 512, 2.2, 0), (320, 832, 2.2, 1)])   # 64 and 65 blocks: one wave sums, sixteen
def test_samples_of_a_partial_last_block_match_the_oracle(swmi, oracle, n0, n1, T, rule):
    """A last block row of few rows leaves tiles without rows; the sample reads nothing past the lattice for them (their
    unused row below the tile used to be read beyond the end of the spin array)."""
    print(f"partial block samples {n0}x{n1} T {T} rule {rule}", flush=True)
    ref = oracle.PerSite(n0, n1, T, seed=6, flip_rule=rule)
    with swmi.Engine(swmi.LatticeConfig(n0, n1, T, seed=6, flip_rule=rule, max_samples=8)) as e:
        e.run(12, 3)
        want = []
        for k in range(12):
            ref.sweep()
            if k % 3 == 2:
                want.append(oracle.observables(n0, n1, ref.spins))
        E, M = e.series()
        assert list(zip(E.tolist(), M.tolist())) == want
        e.spins()   # no flip pending any more
        e.sample()
        assert e.energy_magnetization() == want[-1] and e.moments()[0] == 5 and e.error_flags() == 0
