"""The resident PPCG kernel's source on the CPU (tests/wavefront: a fibre per
lane, one workgroup at a time until all its lanes wait), with the workgroups
in the orders that bring out what one of them must not do before another has
read its cells: every order gives the oracle's fields and values, bit for bit.

A run that starts with p = z + beta p reads its neighbours' p from memory at
its start, so no workgroup may write its own p before that: the last one to
arrive runs on at once, and the others only then read.
"""
from __future__ import annotations

import ctypes
import re
import subprocess

import numpy as np
import pytest

from conftest import REPO
from tealeaf_cuda_amd import Engine
from tealeaf_cuda_amd import runtime as rt

from test_gpu_parity import _prepare, _randomise

HERE = REPO / "tests" / "wavefront"
CSRC = REPO / "tealeaf_cuda_amd" / "csrc"
FIELDS = [rt.FIELD_U, rt.FIELD_P, rt.FIELD_R, rt.XFIELD_Z, rt.XFIELD_KX, rt.XFIELD_KY, rt.XFIELD_RSTORE, rt.FIELD_SD,
          rt.XFIELD_RTEMP, rt.XFIELD_UTEMP]
ALPHAS, BETAS = [0.3, 0.5, 0.7], [1.1, 0.9, 0.8]
NEVER = [-1.0, 1e9, -1.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0]
PREC = {"none": 1, "jac_diag": 2, "jac_block": 3}
_D = ctypes.POINTER(ctypes.c_double)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """resident.hip without its launches, compiled for the CPU."""
    folder = tmp_path_factory.mktemp("wavefront")
    text = (CSRC / "resident.hip").read_text()
    head, rest = text.split("// Picks the kernel of a preconditioner and number of strips.")
    plan = rest[rest.index("}  // namespace\n\nbool plan_tiles"):rest.index("template <typename T>\nhipError_t launch_cg")]
    # (empty asm statements only steer the GPU compiler's registers)
    source = re.sub(r'asm(?: volatile)?\(""[^;]*\);', "", head + plan + "}  // namespace res\n}  // namespace tea\n")
    (folder / "resident_kernels.inc").write_text(source)
    so = folder / "libwavefront.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-pthread", "-ffp-contract=off", "-w",
                    f"-I{HERE}", f"-I{CSRC}", f"-I{folder}", "-o", str(so), str(HERE / "wavefront.cpp")], check=True)
    return ctypes.CDLL(str(so))


@pytest.mark.parametrize("order", [[0, 1], [1, 0]])
@pytest.mark.parametrize("prec", sorted(PREC))
@pytest.mark.parametrize("nx,ny,tiles", [(70, 63, (2, 1)), (20, 120, (1, 2))])
def test_order_of_workgroups(nx, ny, tiles, prec, order, kernels, oracle_so, oracle_env, tmp_path):
    oracle_env("dot2")
    e = Engine(oracle_so)
    try:
        _prepare(e, tmp_path, "ppcg", prec, nx=nx, ny=ny, halo=2)
        _randomise((e,), seed=1)
        e.cg_init()
        e.ppcg_init_constants(ALPHAS, BETAS)
        _randomise((e,), seed=2)
        fields = [e.get_field(fid) for fid in FIELDS]
        its, steps = 2, 3
        table = (_D * len(fields))(*[a.ctypes.data_as(_D) for a in fields])
        history, end = np.zeros(4 * its), ctypes.c_double()
        at_ur, shape = ctypes.c_int(), (ctypes.c_int * 2)()
        coef = np.array(ALPHAS + BETAS)
        n = kernels.ppcg_resident(PREC[prec], nx, ny, 2, 2, (ctypes.c_int * 2)(*order), table, 1,
                                  ctypes.c_double(0.45), ctypes.c_double(0.8), ctypes.c_double(1.7),
                                  coef.ctypes.data_as(_D), steps, its, history.ctypes.data_as(_D),
                                  ctypes.byref(at_ur), ctypes.byref(end), shape)
        assert n == its and tuple(shape) == tiles
        want, want_at_ur, want_end = e.ppcg_run(False, True, 0.45, 0.8, 1.7, steps, its, NEVER)
        assert [tuple(history[4 * k:4 * k + 4]) for k in range(n)] == want
        assert (bool(at_ur.value), end.value) == (want_at_ur, want_end)
        for fid, a in zip(FIELDS, fields):
            if fid != rt.XFIELD_Z:       # (owed by the kernel: z = utemp)
                assert np.array_equal(a, e.get_field(fid), equal_nan=True), f"field {fid}"
    finally:
        e.finalize()
