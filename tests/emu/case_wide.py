"""Emulator cases (TEST INFRASTRUCTURE ONLY): tests/wide_cases.py on a sparse mapping of
the process, of which only the pages of the blocks are ever touched.
Usage: python case_wide.py <stride | deep> <ps>"""
import ctypes
import mmap
import sys

import numpy as np

from emu_harness import Block, emu_lib
import wide_cases as w

MAP_NORESERVE = 0x4000   # linux, not in this mmap module


def run(geom, ps):
    E = emu_lib("emu_lapack")
    rows, cn, _ = w.GEOM[geom]
    big = np.frombuffer(mmap.mmap(-1, rows * cn * 8, mmap.MAP_PRIVATE | mmap.MAP_ANONYMOUS | MAP_NORESERVE), np.float64)

    def upload(a):
        b = Block(a.nbytes)
        b.write(a)
        return b.addr, b

    def lib(entry, batch, args, hint):
        rc = getattr(E, "blasfeo_amd_%s_batched" % entry)(ps, batch, ctypes.c_void_p(args), w.hint(hint), None)
        assert rc == 0, E.emu_last_error()

    for op in w.OPS:
        print("emu wide %s %s ps=%d" % (geom, op, ps), flush=True)
        if op == "ric_trf" and geom == "deep":
            continue   # its matrices have no row offset
        store = w.Store(ps, geom, big.ctypes.data, big.__setitem__, big.__getitem__)
        for k, v in w.knobs(op).items():
            assert E.blasfeo_amd_tune_set(k.encode(), 0, v) == 0
        w.run(op, ps, geom, store, upload, lib)
        for k in w.knobs(op):
            E.blasfeo_amd_tune_set(k.encode(), 0, 0)
    print("ok", flush=True)


if __name__ == "__main__":
    run(sys.argv[1], int(sys.argv[2]))
