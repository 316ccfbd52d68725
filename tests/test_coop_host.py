"""The cooperative block kernels (brams_amd/csrc/rodas3_coop.h) emulated on
the host (tests/host_kernels/coop_host.cpp: a thread for every lane of every
wave) against the oracle's step: attempts, accepted sub-steps, mask and
threshold counts equal, FP32 outputs within a few units in the last place
(the waves' sums run in another order than the oracle's).  One-cell blocks,
blocks of several cells, a block of two halves, RODAS3 and ROS2."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import oracle_lib
from brams_amd.mechanism import load_mechanism
from brams_amd.workload import Grid, make_workload, tolerances

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HERE = os.path.dirname(os.path.abspath(__file__))
MECH = load_mechanism()
CLANG = os.environ.get("HOST_CLANG", "/opt/rocm/llvm/bin/clang++")


@pytest.fixture(scope="module")
def coop_host(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("coop") / "libcoophost.so")
    subprocess.run([CLANG, "-O1", "-std=c++17", "-shared", "-fPIC", "-pthread",
                    "-I", os.path.join(HERE, "host_kernels"), "-I", os.path.join(ROOT, "brams_amd", "csrc"),
                    "-o", lib, os.path.join(HERE, "host_kernels", "coop_host.cpp")], check=True)
    return C.CDLL(lib)


def run(coop_host, wl, atol, rtol, ros2):
    g = wl["grid"]

    def f(a):
        return np.ascontiguousarray(np.asarray(a).ravel(order="F"))

    sc = np.ascontiguousarray(np.stack([f(x) for x in wl["sc_p"]]))
    w = np.array([s.weight for s in MECH.species], np.float32)
    tr = np.array([1 if s.transported else 0 for s in MECH.species], np.int32)
    dt = np.array(wl["last_accepted_dt"], np.float64)
    nblk = len(wl["block_end"])
    start = np.concatenate([[0], np.cumsum(wl["block_end"])]).astype(np.int32)
    counts = np.zeros(4 * nblk + 1, np.int32)
    mw = np.zeros(32, np.uint32)
    pp, pi0, th, rv, jp = f(wl["pp"]), f(wl["pi0"]), f(wl["theta"]), f(wl["rv"]), f(wl["jphoto"])
    at, rt = np.ascontiguousarray(atol, np.float64), np.ascontiguousarray(rtol, np.float64)

    def P(a):
        return a.ctypes.data_as(C.c_void_p)

    coop_host.coop_step_host(1 if ros2 else 0, g.m1, g.m2, g.m3, C.c_float(g.dtlt), nblk, P(start), P(pp), P(pi0),
                             P(th), P(rv), P(jp), P(w), P(tr), P(sc), P(dt), P(at), P(rt), P(counts), P(mw))
    return sc, dt, counts, mw, f


# blocks of 1, 6 and 65 cells, and two blocks of 66
@pytest.mark.parametrize("nx,ny,nz", [(1, 1, 1), (3, 2, 1), (13, 5, 1), (11, 6, 2)])
@pytest.mark.parametrize("solver", ["rodas3", "ros2"])
def test_blocks_match_oracle(coop_host, nx, ny, nz, solver):
    wl = make_workload(Grid(nx, ny, nz, dtlt=30.0), seed=nx, sza="random")
    atol, rtol = tolerances("reference")
    hs, st, mask, rc = oracle_lib.run_oracle(wl, atol, rtol, **({"solver": "ros2"} if solver == "ros2" else {}))
    nblk = len(wl["block_end"])
    oatt, osub = oracle_lib.block_counts(nblk)
    sc, dt, counts, mw, f = run(coop_host, wl, atol, rtol, solver == "ros2")
    ref = np.stack([f(x) for x in hs.sc_p])
    assert rc == 0 and not counts[2 * nblk:3 * nblk].any()
    assert np.array_equal(counts[:nblk], oatt) and np.array_equal(counts[nblk:2 * nblk], osub)
    # half an ulp of the FP32 output where a sum's rounding crosses it
    np.testing.assert_allclose(sc, ref, rtol=1.2e-7, atol=0)
    np.testing.assert_allclose(dt, hs.last_dt, rtol=1e-10)
    if solver == "rodas3":
        assert counts[3 * nblk:4 * nblk].sum() == oracle_lib.block_thresholds(nblk)[0]
        assert counts[4 * nblk] == st.order_threshold_pivots
        assert sum(bin(int(x)).count("1") for x in mw) == st.mask_nnz
