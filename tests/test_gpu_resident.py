"""Small lattices are swept whole in one workgroup (k_resident) unless the caller asks for a tile height; the tiled
kernels give the same chain. Both against the oracle, at the edges of what one workgroup takes: one and sixteen tile
columns, strips of one to sixteen rows, a strip count that leaves waves idle, padded and narrow rows, the largest
lattice and the first one past it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TC = 2.2691853

EXTENTS = [(64, 2), (64, 64), (64, 256), (192, 64), (1024, 16), (128, 128), (126, 100), (130, 18), (100, 162), (32, 32), (32, 512),
           (16, 6), (48, 34), (2, 2), (30, 200), (64, 258),
           (4, 2048), (4, 2064)]   # below 16 columns: the last lattice of eight rows per strip and the first past it


@pytest.mark.parametrize("n0,n1", EXTENTS)
@pytest.mark.parametrize("tile_rows", [0, 16])
@pytest.mark.parametrize("rule", [0, 1])
def test_sweeps_labels_samples_and_generator_match_the_oracle(swmi, oracle, n0, n1, tile_rows, rule):
    print(f"resident {n0}x{n1} tile_rows {tile_rows} rule {rule}", flush=True)
    T = 2.0 + 0.3 * ((n0 + n1) % 3)
    ref = oracle.PerSite(n0, n1, T, seed=n0 + n1, spin_seed=3, flip_rule=rule)
    cfg = swmi.LatticeConfig(n0, n1, T, seed=n0 + n1, spin_seed=3, tile_rows=tile_rows, flip_rule=rule, max_samples=8)
    with swmi.Engine(cfg) as e:
        _, labels = ref.sweep(record=True)
        e.sweep(1)
        np.testing.assert_array_equal(e.labels(), labels, err_msg="labels, sweep 1")
        np.testing.assert_array_equal(e.spins(), ref.spins, err_msg="spins, sweep 1")
        e.run(20, 5)   # across rotations at updates 15, 30
        samples = []
        for k in range(20):
            _, labels = ref.sweep(record=True)
            if k % 5 == 4:
                samples.append(oracle.observables(n0, n1, ref.spins))
        E, M = e.series()
        assert list(zip(E.tolist(), M.tolist())) == samples
        np.testing.assert_array_equal(e.labels(), labels, err_msg="labels, sweep 21")
        np.testing.assert_array_equal(e.spins(), ref.spins, err_msg="spins, sweep 21")
        st = e.rng_state()
        np.testing.assert_array_equal(st["states"], ref.states)
        np.testing.assert_array_equal(st["rot"], ref.rot)
        assert st["iteration"] == 42 and e.error_flags() == 0
        n = float(n0 * n1)
        ev = [-s[0] / n for s in samples]
        assert e.moments()[0] == 4 and e.moments()[1] == ((ev[0] + ev[1]) + ev[2]) + ev[3]


@pytest.mark.parametrize("n0,n1", [(64, 64), (128, 128), (100, 100), (32, 32)])
@pytest.mark.parametrize("rule", [0, 1])
def test_the_two_paths_take_over_from_each_other(swmi, oracle, n0, n1, rule):
    """Recording bonds runs the tiled kernels, so switching it moves a chain between the paths, with a flip pending
    and with generator states of an earlier update; checkpoints pass between them too."""
    print(f"resident and tiled {n0}x{n1} rule {rule}", flush=True)
    ref = oracle.PerSite(n0, n1, TC, seed=7, spin_seed=4, flip_rule=rule)

    def advance(k):
        for _ in range(k):
            ref.sweep()

    with swmi.Engine(swmi.LatticeConfig(n0, n1, TC, seed=7, spin_seed=4, flip_rule=rule)) as e:
        for k in (3, 6, 1, 9):
            e.record_bonds(True)
            e.sweep(k)           # tiled: leaves its last flip pending
            e.record_bonds(False)
            advance(k)
            if k == 1:
                e.sample()       # a sample of a pending flip by the resident path
                np.testing.assert_array_equal(e.spins(), ref.spins)
            e.sweep(k)
            advance(k)
            np.testing.assert_array_equal(e.spins(), ref.spins, err_msg=f"after {k} and {k} sweeps")
        ck = e.checkpoint()
        assert e.error_flags() == 0
    with swmi.Engine(swmi.LatticeConfig(n0, n1, 2.0, seed=1, tile_rows=16)) as tiled:
        tiled.restore(ck)
        tiled.sweep(8)
        advance(8)
        np.testing.assert_array_equal(tiled.spins(), ref.spins, err_msg="tiled, from a resident lattice's checkpoint")
        ck = tiled.checkpoint()
    with swmi.Engine(swmi.LatticeConfig(n0, n1, 2.0, seed=1)) as e:
        e.restore(ck)
        e.sweep(8)
        advance(8)
        np.testing.assert_array_equal(e.spins(), ref.spins, err_msg="resident, from a tiled lattice's checkpoint")
        assert e.error_flags() == 0


@pytest.mark.parametrize("rule", [0, 1])
def test_lattices_of_every_kind_in_one_launch_match_the_oracle(swmi, oracle, rule):
    """k_resident_mixed: all the extents above in one engine, their labels, samples and generators included."""
    extents = [x for x in EXTENTS if x not in ((64, 258), (4, 2064))]
    print(f"resident, every kind, rule {rule}", flush=True)
    T = [2.0 + 0.1 * (i % 6) for i in range(len(extents))]
    refs = [oracle.PerSite(n0, n1, T[i], seed=i, spin_seed=3, flip_rule=rule) for i, (n0, n1) in enumerate(extents)]
    with swmi.Engine([swmi.LatticeConfig(n0, n1, T[i], seed=i, spin_seed=3, flip_rule=rule, max_samples=8)
                      for i, (n0, n1) in enumerate(extents)]) as e:
        e.sweep(3)
        e.run(20, 5)
        for i, ((n0, n1), ref) in enumerate(zip(extents, refs)):
            samples = []
            for k in range(23):
                _, labels = ref.sweep(record=True)
                if k >= 3 and (k - 3) % 5 == 4:
                    samples.append(oracle.observables(n0, n1, ref.spins))
            E, M = e.series(i)
            assert list(zip(E.tolist(), M.tolist())) == samples, (n0, n1)
            np.testing.assert_array_equal(e.labels(i), labels, err_msg=f"labels {n0}x{n1}")
            np.testing.assert_array_equal(e.spins(i), ref.spins, err_msg=f"spins {n0}x{n1}")
            st = e.rng_state(i)
            np.testing.assert_array_equal(st["states"], ref.states)
            np.testing.assert_array_equal(st["rot"], ref.rot)
            assert e.error_flags(i) == 0


def test_schedules_and_long_loops_of_a_mixed_engine(swmi):
    """Resident, tiled and scheduled lattices in one engine equal their lone runs; loops longer than one launch."""
    print("resident mixed engine", flush=True)
    cfgs = [swmi.LatticeConfig(64, 64, 2.1, seed=1, max_samples=200), swmi.LatticeConfig(256, 256, 2.2, seed=2, max_samples=200),
            swmi.LatticeConfig(128, 128, 2.3, seed=3, max_samples=200), swmi.LatticeConfig(100, 100, 2.4, seed=4, max_samples=200),
            swmi.LatticeConfig(32, 32, 2.5, seed=5, max_samples=200)]
    plans = [(1130, 30), (700, 100), (640, 0), (55, 10), (0, 20)]

    def drive(engine, lattices):
        for i, k in enumerate(lattices):
            engine.set_schedule(i, sweeps=plans[k][0], warmup=plans[k][1], n_sep=10)
        engine.run_scheduled(1200, 10)
        engine.sweep(30)
        return [(engine.spins(i), engine.moments(i), engine.series(i), engine.progress(i)) for i in range(len(lattices))]

    with swmi.Engine(cfgs) as e:
        got = drive(e, range(5))
    for k, c in enumerate(cfgs):
        for rows in (0, 16):
            c.tile_rows = rows
            with swmi.Engine(c) as alone:
                spins, moments, series, progress = drive(alone, [k])[0]
            np.testing.assert_array_equal(spins, got[k][0], err_msg=f"lattice {k} tile_rows {rows}")
            np.testing.assert_array_equal(moments, got[k][1])
            np.testing.assert_array_equal(series, got[k][2])
            assert progress == got[k][3]
