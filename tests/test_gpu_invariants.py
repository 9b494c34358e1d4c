"""Labels that break an invariant of the engine are reported through the error flags, not followed: the kernels that read
them get buffers in which one label or count is out of its range (the engine itself never writes such a one)."""
import ctypes

import numpy as np
import pytest

from raw_lattice import APPLIED, EDGE, ERRORS, ITERATION, RawLattice

pytestmark = pytest.mark.gpu

u32, i32, flag = ctypes.c_uint32, ctypes.c_int32, ctypes.c_bool
N_SLOTS = 252   # most boundary sites of a block of 64 columns and 64 rows


def _two_by_two(swmi):
    """128 x 128 in four blocks, each with one cluster on its whole edge: slot 0, rooted at the block's first site."""
    r = RawLattice(swmi, 128, 128, 16)
    entry = (EDGE | r.g.qcap) << 16
    r.a["ecol"][:] = entry
    r.a["erow"][:] = entry
    r.a["edge_count"][::4] = 1
    return r


def _label(r, index, edge=True, root=0):
    return ((EDGE if edge else 0) | index) << 16 | root


@pytest.mark.parametrize("fault", ["none", "bonds", "slot", "slot on a bond", "last slot", "unnamed slot", "stray label", "unflagged on a bond"])
def test_join_reports_broken_labels(swmi, fault):
    print(f"join with {fault}", flush=True)
    r = _two_by_two(swmi)
    bad = fault not in ("none", "bonds", "last slot", "slot")   # (a label that nothing joins is not looked at)
    if fault != "none":
        r.a["bbits"][::5] = 2 ** 64 - 1     # every down bond
        r.a["bbits"][1::5] = 0xFFFF         # right bonds of each block's first tile
    if fault in ("slot", "slot on a bond"):   # row 40 of the last column has no bond, row 3 has one
        r.a["ecol"][2, 1, 3 if "bond" in fault else 40] = _label(r, r.g.qcap + 256)
    if fault == "last slot":                # slots 0 .. 251, each on one site of the block's edge
        sites = [("ecol", 1, 0, y) for y in range(64)] + [("ecol", 1, 1, y) for y in range(64)] + \
                [("erow", 1, 0, x) for x in range(1, 63)] + [("erow", 1, 1, x) for x in range(1, 63)]
        for s, at in enumerate(sites):
            r.a[at[0]][at[1:]] = _label(r, r.g.qcap + s, root=64 * at[3] if at[0] == "ecol" else at[3])
        assert len(sites) == N_SLOTS
        r.a["edge_count"][4] = N_SLOTS
        r.a["bbits"][:] = 0
    if fault == "unnamed slot":             # the node holds what the LDS held before: the chase ends, whatever that was
        r.a["edge_count"][8] = 200
    if fault == "stray label":              # a first-row lane that holds no site's slot names a root past the block
        r.a["erow"][1, 0, 7] = _label(r, 64 * 64 + 1, edge=False)
        r.a["bbits"][:] = 0
    if fault == "unflagged on a bond":
        r.a["ecol"][1, 0, 2] = _label(r, 5, edge=False)
    state = r.launch("_ZN4swmi10LaunchJoinEPKNS_7LatDescEPKjjjP12ihipStream_t", [u32, u32], 1, 4)
    r.close()
    assert state[ERRORS] == (1 if bad else 0) or fault == "unnamed slot"
    assert state[ITERATION] == 2


def _pending(swmi):
    """128 x 128 in four blocks, the last sweep's flip pending: every site a cluster of its own block's root 0."""
    r = RawLattice(swmi, 128, 128, 16)
    r.a["state"][[ITERATION, APPLIED]] = 4, 2
    r.a["aux"][0] = 4
    return r


# (label, is it in its range): roots of a block of 64 x 64 sites, then slots
LABELS = [(4095, True), (4096, False), (0x7FFF, False), ("slot 0", True), ("slot 251", True), ("last slot", True), ("past the slots", False),
          (EDGE, False)]


@pytest.mark.parametrize("label,good", LABELS)
@pytest.mark.parametrize("reader", ["sample", "resident"])
def test_readers_of_a_pending_flip_report_broken_labels(swmi, label, good, reader):
    print(f"pending flip, label {label}, {reader}", flush=True)
    r = _pending(swmi)
    slots = 4 * r.g.edge_cap
    index = {"slot 0": 0, "slot 251": 251, "last slot": slots - 1, "past the slots": slots}
    r.a["local"][128 * 100 + 77] = EDGE | (r.g.qcap + index[label]) if label in index else label
    if reader == "sample":
        state = r.launch("_ZN4swmi17LaunchObservablesEPKNS_7LatDescEPKjjjP12ihipStream_t", [u32, u32], 4, 0)
    else:
        state = r.launch("_ZN4swmi14LaunchResidentEPKNS_7LatDescEPKjjjjbbbbjjiP12ihipStream_t",
                         [u32, u32, u32, flag, flag, flag, flag, u32, u32, i32], 1, 16384, 16, True, True, False, False, 1, 1, -1)
    r.close()
    assert state[ERRORS] == (0 if good else 1)
    assert state[ITERATION] == (4 if reader == "sample" else 6)
