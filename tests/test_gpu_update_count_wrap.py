"""The lcg32 update count is a 32-bit number that a chain of 2^31 sweeps wraps (a few hours at 64^2); a lattice without a
schedule goes on. The last update before the wrap and the first after it both rotate (2^32 - 1 and 0 are multiples of 15)
and fall into one sweep. A checkpoint with the count set just below the wrap gets there in a few sweeps; the oracle
starts from the same count."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

HEADER = 64   # bytes before the arrays of a checkpoint


def _near_the_wrap(checkpoint, n_padded, iteration):
    data = bytearray(checkpoint)
    state = HEADER + n_padded * (1 + 4) + n_padded // 64 * (3 * 8 + 4)   # spins, states, selector planes, rotations
    assert int.from_bytes(data[state:state + 4], "little") == 0
    data[state:state + 4] = iteration.to_bytes(4, "little")
    return bytes(data)


@pytest.mark.parametrize("n0,n1,tile_rows", [(64, 64, 0), (100, 100, 0), (32, 32, 0), (64, 64, 16), (128, 320, 0), (130, 300, 0), (32, 1030, 0),
                                             (1024, 1100, 0), (128, 128, 64)])
@pytest.mark.parametrize("rule", [0, 1])
def test_sweeps_across_the_wrap_match_the_oracle(swmi, oracle, n0, n1, tile_rows, rule):
    print(f"update count wrap {n0}x{n1} tile_rows {tile_rows} rule {rule}", flush=True)
    first = 2 ** 32 - 12
    T = 2.2691853
    ref = oracle.PerSite(n0, n1, T, seed=6, spin_seed=2, flip_rule=rule)
    ref.iteration.value = first
    with swmi.Engine(swmi.LatticeConfig(n0, n1, T, seed=6, spin_seed=2, tile_rows=tile_rows, flip_rule=rule)) as e:
        pitch, _ = e.layout()
        e.restore(_near_the_wrap(e.checkpoint(), pitch * n1, first))
        for sweeps in (5, 1, 20):   # to the wrap, the sweep of two rotations, on across the next rotations
            e.sweep(sweeps)
            for _ in range(sweeps):
                ref.sweep()
            np.testing.assert_array_equal(e.spins(), ref.spins, err_msg=f"spins at update {ref.iteration.value}")
            st = e.rng_state()
            np.testing.assert_array_equal(st["states"], ref.states)
            np.testing.assert_array_equal(st["rot"], ref.rot)
            assert st["iteration"] == ref.iteration.value
        assert e.error_flags() == 0
    assert ref.iteration.value == 2 * 26 - 12
    # all of it in one call
    with swmi.Engine(swmi.LatticeConfig(n0, n1, T, seed=6, spin_seed=2, tile_rows=tile_rows, flip_rule=rule)) as e:
        e.restore(_near_the_wrap(e.checkpoint(), pitch * n1, first))
        e.sweep(26)
        np.testing.assert_array_equal(e.spins(), ref.spins)
        assert e.error_flags() == 0
