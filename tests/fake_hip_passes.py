"""Runs in a process of its own (test_host_allocation.py): FP64 passes and CG solves of a one-specimen
hexa8 context on the stand-in runtime, with each allocation of the first pass failing in turn.  Prints a
line per run: rc of the pass, rc of the solve, whether the solve took the bricks."""

import ctypes
import os
import sys

import numpy as np

fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_launches.restype = ctypes.c_char_p
fake.fake_fail.argtypes = [ctypes.c_long]
fake.fake_allocations.restype = ctypes.c_long
sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
from edelweissfe_amd import _lib  # noqa: E402
from edelweissfe_amd.generators.boxgen import generateBox  # noqa: E402

J2 = np.array([210000.0, 0.3, 250.0, 1000.0, 0.0, 0.0])
lib = _lib.load()


def run(failing):
    pm = generateBox(3, 2, 2, 1.0, 1.0, 1.0, elType="C3D8", jitter=0.1, seed=1)
    coords = np.ascontiguousarray(pm.coordinates, dtype=np.float64)
    conn = np.ascontiguousarray(pm.connectivity, dtype=np.int32)
    spec = np.zeros(len(coords), dtype=np.int32)
    d = _lib.MeshDesc(n_nodes=len(coords), n_elements=len(conn), element_type=_lib.EFE_C3D8,
                      material=_lib.EFE_VONMISES, coords=coords.ctypes.data, conn=conn.ctypes.data, n_props=6,
                      props_per_element=0, props=J2.ctypes.data, specimen_of_node=spec.ctypes.data, n_specimens=1)
    ctx = ctypes.c_void_p()
    _lib.check(lib.efe_ctx_create(ctypes.byref(d), ctypes.byref(ctx)), "efe_ctx_create")
    v = [np.zeros(3 * len(coords)) for _ in range(5)]
    time, pnew = (ctypes.c_double * 2)(0.0, 0.0), ctypes.c_double(1.0)

    def one_pass():
        return lib.efe_compute_elements(ctx, None, v[0].ctypes.data, time, 0.0, v[1].ctypes.data, v[2].ctypes.data,
                                        None, None, _lib.EFE_FP64, ctypes.byref(pnew))

    fake.fake_fail(failing)
    rc = one_pass()
    n = fake.fake_allocations()
    fake.fake_fail(-1)
    if rc == 0:
        rc = one_pass()  # and the next one stays with what the first found
    fake.fake_launches()
    o = _lib.SolveOpts(solver=_lib.EFE_SOLVER_CG, precision=_lib.EFE_FP64, max_iter=10, check_every=2, rtol=1e-8)
    info = _lib.SolveInfo()
    rs = lib.efe_linsolve(ctx, v[3].ctypes.data, v[4].ctypes.data, ctypes.byref(o), ctypes.byref(info))
    names = fake.fake_launches().decode()
    init = [k for k in names.splitlines() if "pcg_init_kernel" in k]
    lib.efe_ctx_destroy(ctx)
    print(failing, n, rc, rs, int(any("ELb1E" in k for k in init)), flush=True)


run(-1)
for k in range(int(sys.argv[2])):
    run(k)
