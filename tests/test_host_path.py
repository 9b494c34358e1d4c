"""The engine's host side on a machine without a GPU: libswmi.so over a recorder that stands in for the HIP runtime
(hip_recorder.cpp) and runs no kernel. Checks which kernels a call launches, in which order over the streams, and what it
does when a runtime call fails."""
import subprocess
import sys
import textwrap
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
PRELUDE = """
import ctypes, re, sys
sys.path.insert(0, {root!r})
rec = ctypes.CDLL({recorder!r}, mode=ctypes.RTLD_GLOBAL)
rec.rec_take.restype = ctypes.c_char_p
rec.rec_fail.argtypes = [ctypes.c_char_p, ctypes.c_size_t]
rec.rec_cost.argtypes = [ctypes.c_char_p, ctypes.c_double]
import computational_physics_amd as cpa

def take():
    return rec.rec_take().decode().splitlines()

def fail(name, least=0):
    rec.rec_fail(name.encode(), least)

def launched(lines):
    return [m.group(1) for l in lines for m in [re.match(r"(?:captured )?launch \\\\S*?(k_[a-z_]+?)(?:I|E|P)", l)] if m]
"""


@pytest.fixture(scope="module")
def recorded(tmp_path_factory):
    lib = tmp_path_factory.mktemp("recorder") / "hip_recorder.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-Wno-deprecated-declarations",
                    "-o", str(lib), str(ROOT / "tests" / "hip_recorder.cpp")], check=True, timeout=300)

    def run(script):
        code = PRELUDE.format(root=str(ROOT), recorder=str(lib)).replace("\\\\", "\\") + textwrap.dedent(script)
        got = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
        assert got.returncode == 0, got.stdout[-3000:] + got.stderr[-3000:]

    return run


@pytest.mark.parametrize("call", ["e.sweep(64)", "e.run(640, 10)"])
@pytest.mark.parametrize("failing", ["hipStreamBeginCapture", "hipGraphInstantiate"])
def test_a_failed_call_still_joins_the_resident_stream(recorded, call, failing):
    """A 64^2 lattice is swept on a side stream beside a 256^2 one; whatever fails after its launch, the engine stream
    waits for it before the call returns, so that a later read on that stream sees the sweeps."""
    recorded(f"""
        e = cpa.Engine([cpa.LatticeConfig(64, 64), cpa.LatticeConfig(256, 256)])
        take()
        fail({failing!r})
        try:
            {call}
            raise SystemExit("the call did not fail")
        except cpa.SwmiError:
            pass
        lines = take()
        last = max(i for i, l in enumerate(lines) if "k_resident" in l)
        side = lines[last].rsplit(" ", 1)[1]
        records = [(i, l.split()[2]) for i, l in enumerate(lines) if i > last and l.startswith("record") and l.endswith(" stream " + side)]
        assert records, lines
        at, event = records[-1]
        waits = [l.split()[2] for l in lines[at:] if l.startswith("wait") and l.endswith(" event " + event)]
        assert waits and waits[0] != side, lines
        fail("")
        e.sweep(64)
        assert "k_resident" in launched(take())
    """)


@pytest.mark.parametrize("n0,n1", [(128, 256), (100, 300)])
def test_spins_are_read_back_when_no_device_memory_is_left(recorded, n0, n1):
    """An engine that fills the device still returns its spins: the download then needs no memory there."""
    recorded(f"""
        import numpy as np
        n0, n1 = {n0}, {n1}
        e = cpa.Engine(cpa.LatticeConfig(n0, n1))
        pitch, _ = e.layout()
        data = bytearray(e.checkpoint())
        padded = np.random.default_rng(1).integers(0, 64, pitch * n1).astype(np.uint8)   # spins and selector bits
        data[64:64 + pitch * n1] = padded.tobytes()
        e.restore(bytes(data))
        fail("hipMalloc", 64)
        np.testing.assert_array_equal(e.spins().reshape(n1, n0), padded.reshape(n1, pitch)[:, :n0] & 1)
        fail("")
        take()
        e.spins()
        assert "k_get_spins" in launched(take())
    """)


@pytest.mark.parametrize("untiled_wins", [True, False])
def test_autotuners_measure_and_return_the_untiled_path(recorded, untiled_wins):
    """A lattice that one workgroup sweeps is timed that way too: tile_rows 0 comes back when it is the fastest, and a
    height found faster is what a later lattice of this extent runs with."""
    recorded(f"""
        wins = {untiled_wins}
        rec.rec_cost(b"k_resident", 1.0 if wins else 1e5)
        small = cpa.LatticeConfig(64, 64)
        best, ms = cpa.autotune(small, sweeps=20)
        assert (best == 0) == wins and len(ms) == 7 and best in (0, 1, 2, 4, 8, 16, 32, 64), (best, ms)
        take()
        e = cpa.Engine(small)
        e.sweep(3)
        assert ("k_resident" in launched(take())) == wins
        assert wins or e.tile_rows() == best
        batch = [cpa.LatticeConfig(48, 48), cpa.LatticeConfig(256, 256)]
        best, ms = cpa.autotune_batch(batch, sweeps=20)
        assert (best == 0) == wins and len(ms) == 7 and min(ms) > 0, (best, ms)
        # nothing to sweep untiled: always a height
        assert cpa.autotune(cpa.LatticeConfig(256, 256), sweeps=20)[0] > 0
        assert cpa.autotune_batch([cpa.LatticeConfig(256, 256), cpa.LatticeConfig(512, 320)], sweeps=20)[0] > 0
    """)


@pytest.mark.parametrize("sizes", [[(64, 64)], [(256, 256)], [(2048, 512)], [(64, 64), (32, 32), (256, 256), (2048, 512)]])
def test_time_kernels_times_the_kernels_of_a_sweep(recorded, sizes):
    """The same launches as a sweep loop's, each counted in its figure (one microsecond a launch here)."""
    recorded(f"""
        from collections import Counter
        e = cpa.Engine([cpa.LatticeConfig(n0, n1) for n0, n1 in {sizes}])
        take()
        e.set_graphs(False)
        e.sweep(12)
        want = Counter(launched(take()))
        ms = e.time_kernels(12)
        assert Counter(launched(take())) == want
        parts = [("k_bond_label", "k_resident"), ("k_merge", "k_join"), ("k_resolve",)]
        for figure, names in zip(ms, parts):
            launches = sum(n for k, n in want.items() if k.startswith(names))
            assert abs(figure * 12 - launches * 1e-3) < 1e-6, (ms, want)
    """)


@pytest.mark.parametrize("n0,n1,count,joined", [(64, 64, 512, True), (64, 64, 513, False), (64, 256, 600, True), (64, 128, 600, False),
                                                (256, 256, 600, True), (64, 1088, 1, False), (64, 1024, 1, True)])
def test_many_lattices_of_few_blocks_merge_and_resolve_block_by_block(recorded, n0, n1, count, joined):
    recorded(f"""
        e = cpa.Engine([cpa.LatticeConfig({n0}, {n1}, tile_rows=16) for _ in range({count})])
        take()
        e.sweep(1)
        kernels = launched(take())
        assert kernels == ["k_bond_label", "k_join"] if {joined} else kernels[-1] == "k_resolve" and "k_join" not in kernels, kernels
    """)


@pytest.mark.parametrize("n0,n1,least", [(64, 64, 2560), (34, 6, 2560), (8, 8, 4096), (16, 16, 4096), (32, 32, 0), (128, 8, 0)])
def test_very_many_of_the_smallest_lattices_are_swept_tiled(recorded, n0, n1, least):
    recorded(f"""
        for count in ({least} - 1, {least}) if {least} else (4200,):
            e = cpa.Engine([cpa.LatticeConfig({n0}, {n1}) for _ in range(count)])
            take()
            e.sweep(2)
            assert ("k_resident" in launched(take())) == (count != {least}), count
    """)


def _routes(recorded, sizes, want):
    """Kernels of one sweep of an engine of these lattices against `want`, a list of name and grid pairs."""
    recorded(f"""
        e = cpa.Engine([cpa.LatticeConfig(n0, n1) for n0, n1 in {sizes}])
        take()
        e.sweep(1)
        lines = [l for l in take() if l.startswith("launch")]
        got = sorted((k, int(re.search(r" grid (\\d+)", l).group(1))) for k, l in zip(launched(lines), lines))
        assert got == sorted({want}), got
    """)


def test_resident_lattices_of_several_kinds_share_one_launch(recorded):
    small = [(32, 32), (64, 64), (128, 128), (100, 100), (48, 48)]
    _routes(recorded, small, [("k_resident_mixed", 5)])
    _routes(recorded, [(64, 64)] * 7, [("k_resident", 7)])
    _routes(recorded, [(64, 64)] * 200 + [(128, 128)] * 56, [("k_resident_mixed", 256)])
    _routes(recorded, [(64, 64)] * 200 + [(128, 128)] * 57, [("k_resident", 200), ("k_resident", 57)])
    # one tiled class beside them changes nothing
    _routes(recorded, small + [(512, 512)], [("k_resident_mixed", 5), ("k_bond_label", 64), ("k_merge", 64), ("k_resolve", 64)])


def test_small_lattices_go_along_with_a_tiled_class_where_there_are_several(recorded):
    tiled = [("k_bond_label", 72), ("k_merge", 72), ("k_resolve", 72), ("k_bond_label", 264), ("k_merge", 264), ("k_resolve", 264)]
    # 128^2 joins 512^2 (4 + 64 blocks) and 100^2 joins 1000^2 (4 + 256); 32^2 has no tiled class of its own
    _routes(recorded, [(128, 128), (100, 100), (512, 512), (1000, 1000)], tiled)
    _routes(recorded, [(128, 128), (100, 100), (512, 512), (1000, 1000), (32, 32)], tiled + [("k_resident", 1)])
    # more blocks than the tiled class has: resident
    _routes(recorded, [(128, 128)] * 17 + [(512, 512), (1000, 1000)],
            [("k_resident", 17), ("k_bond_label", 64), ("k_merge", 64), ("k_resolve", 64), ("k_bond_label", 256), ("k_merge", 256), ("k_resolve", 256)])
