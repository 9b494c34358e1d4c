"""One lattice's device buffers under the kernels' launch wrappers (csrc/swmi_internal.h), for tests that hand a kernel
labels the engine would never write: the kernels report those through the lattice's error flags."""
import ctypes

import numpy as np

from test_zz_no_alloc import _Hip

u32, u64, vp = ctypes.c_uint32, ctypes.c_uint64, ctypes.c_void_p


class Geometry(ctypes.Structure):
    _fields_ = [(f, u32) for f in ("pitch", "tw", "rpw", "twr", "tiles_x", "blocks_y", "nwr_y", "n_blocks", "edge_cap", "ecol_stride",
                                   "halo_stride", "elast", "qcap", "fsw")] + [("vlast", u64)]


class LatDesc(ctypes.Structure):
    _fields_ = [(f, vp) for f in ("spins", "rng", "aux", "masks", "rot", "local", "parent", "cpar", "bbits", "state", "bond_dump", "bond_in",
                                  "partials", "edge_count", "ecol", "erow")] + \
               [(f, u32) for f in ("ecol_stride", "edge_cap", "qcap", "fsw", "n0", "n1", "n0v", "elast")] + [("vlast", u64)] + \
               [(f, u32) for f in ("tw", "rpw", "twr", "tiles_x", "blocks_y", "nwr_y", "threshold", "block_base", "n_blocks", "flip_rule", "seed")] + \
               [("fbits", vp), ("halo", vp), ("halo_stride", u32)]


ITERATION, ERRORS, IT_END, ACTIVE, APPLIED = 0, 3, 4, 5, 10   # words of LatState
STATE_WORDS = 24
EDGE = 0x8000


class RawLattice:
    def __init__(self, swmi, n0, n1, tile_rows):
        self.lib = swmi.load_library()
        self.hip = _Hip()
        geometry_of, desc_of = self.lib._ZN4swmi10GeometryOfEjjj, self.lib._ZN4swmi12GeometryDescERKNS_8GeometryEjj
        geometry_of.restype, geometry_of.argtypes = Geometry, [u32] * 3
        desc_of.restype, desc_of.argtypes = LatDesc, [ctypes.POINTER(Geometry), u32, u32]
        self.g = geometry_of(n0, n1, tile_rows)
        self.d = desc_of(ctypes.byref(self.g), n0, n1)
        assert self.d.n0v == n0 and self.d.n1 == n1 and self.d.halo_stride == self.g.halo_stride   # the mirrored layouts hold
        g = self.g
        self.n = n0 * n1
        self.a = {"spins": np.zeros(self.n, np.uint8), "rng": np.zeros(self.n, np.uint32), "aux": np.zeros(2, np.uint32),
                  "rot": np.zeros(self.n // 64, np.uint32), "local": np.zeros(self.n, np.uint16),
                  "cpar": np.zeros(4 * g.edge_cap * g.n_blocks, np.uint64), "bbits": np.zeros(5 * g.n_blocks, np.uint64),
                  "state": np.zeros(STATE_WORDS, np.uint32), "partials": np.zeros(2 * g.n_blocks, np.int32),
                  "edge_count": np.zeros(4 * g.n_blocks, np.uint32), "ecol": np.zeros((g.n_blocks, 2, g.ecol_stride), np.uint32),
                  "erow": np.zeros((g.n_blocks, 2, 64), np.uint32), "fbits": np.zeros(g.fsw * g.n_blocks, np.uint32),
                  "halo": np.zeros(2 * g.n_blocks * g.halo_stride, np.uint8)}
        self.a["state"][[IT_END, ACTIVE]] = 0xFFFFFFFF, 1
        self.memory = []

    def launch(self, name, argtypes, *args):
        """Uploads the arrays and the descriptor, launches name(descriptors, list, *args, stream 0) and returns the state words.
        The list names lattice 0 once per block: it serves the kernels that read one entry per lattice and those that read
        one per block."""
        for field, array in self.a.items():
            p = self.hip.malloc(array.nbytes)
            self.memory.append(p)
            self.hip.h2d(p, array)
            setattr(self.d, field, p.value)
        zero = np.zeros(self.g.n_blocks, np.uint32)
        desc, slots = self.hip.malloc(ctypes.sizeof(LatDesc)), self.hip.malloc(zero.nbytes)
        self.memory += [desc, slots]
        self.hip.h2d(desc, np.frombuffer(bytes(self.d), np.uint8).copy())
        self.hip.h2d(slots, zero)
        fn = getattr(self.lib, name)
        fn.restype, fn.argtypes = None, [vp, vp, *argtypes, vp]
        fn(desc, slots, *args, None)
        self.hip.check(self.hip.lib.hipDeviceSynchronize(), name)
        out = np.zeros(STATE_WORDS, np.uint32)
        self.hip.d2h(out, vp(self.d.state))
        return out

    def close(self):
        for p in self.memory:
            self.hip.lib.hipFree(p)
