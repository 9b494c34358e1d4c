"""Bond fields of small lattices are labelled by one workgroup in one launch (k_label_whole); larger ones by the tiled
kernels. Against the oracle, at the edges of what one workgroup takes: narrow and padded rows, one and sixteen tile
columns, strips of one to sixteen rows, idle waves, the largest lattice and the first past it; empty, full and critical
fields."""
import ctypes

import numpy as np
import pytest

from test_zz_no_alloc import _bonds, _Hip

pytestmark = pytest.mark.gpu

EXTENTS = [(2, 2), (16, 6), (6, 8), (32, 32), (30, 200), (32, 512), (48, 34), (62, 2), (64, 2), (64, 64), (64, 256), (64, 258), (66, 50),
           (126, 100), (128, 128), (130, 18), (192, 64), (1000, 6), (1024, 16), (1026, 14),
           # tiled: partial and padded blocks, 16, 8 and 4 waves per block, narrow rows
           (300, 300), (64, 1000), (512, 320), (1000, 1350), (1536, 1024), (2048, 1024), (1100, 3000), (32, 2048), (30, 1000), (16, 4096)]


def test_small_bond_fields_match_the_oracle(swmi, oracle):
    hip = _Hip()
    stream = ctypes.c_void_p()
    hip.check(hip.lib.hipStreamCreate(ctypes.byref(stream)), "hipStreamCreate")
    rng = np.random.default_rng(5)
    n_max = max(n0 * n1 for n0, n1 in EXTENTS)
    d_bonds, d_labels = hip.malloc(n_max), hip.malloc(4 * n_max)
    try:
        for n0, n1 in EXTENTS:
            print(f"whole labelling {n0}x{n1}", flush=True)
            for density in (0.0, 0.4, 0.5, 0.7, 1.0):
                bonds = _bonds(rng, n0, n1, density)
                hip.h2d(d_bonds, bonds)
                swmi.label_bonds_noalloc(d_bonds.value, n0, n1, d_labels.value, stream.value)
                hip.check(hip.lib.hipStreamSynchronize(stream), "hipStreamSynchronize")
                got = np.empty(n0 * n1, dtype=np.uint32)
                hip.d2h(got, d_labels)
                np.testing.assert_array_equal(got, oracle.label(n0, n1, bonds), err_msg=f"{n0}x{n1} density {density}")
    finally:
        hip.lib.hipFree(d_bonds)
        hip.lib.hipFree(d_labels)
        hip.lib.hipStreamDestroy(stream)
