"""GPU parity of the QSSA solver (chem_spack_qssa.f90, CHEMISTRY=1) against
the oracle's QSSA through the C-ABI.

The step writes tendencies only, so the check is on the new mixing ratio
they imply, x = sc_p + sc_t dtlt, per cell and species: within rel 1e-6 of
the oracle's, plus 1e-7 of the old value (the REAL tendency's rounding), plus
the conditioning of the reference's own recurrence.  That recurrence,
P/ybid + (y - P/ybid) e, loses about one rounding of max(|P/ybid|, |y|) per
sub-step: where L is tiny, P/ybid is huge and the result is defined only to
itchim x 4 eps x that amount (1e-13 of it is allowed; computed from the
oracle's P and L for the cells outside the plain bound).
"""
import math

import numpy as np
import pytest

import oracle_lib as O
from brams_amd.mechanism import load_mechanism
from brams_amd.workload import Grid, make_workload

pytestmark = pytest.mark.gpu
MECH = load_mechanism()
NS = MECH.nspecies
ITCHIM = 75


def _gpu(wl, itchim=ITCHIM, sc_t=None):
    from brams_amd import abi
    from brams_amd.chem import DeviceStep
    ds = DeviceStep(wl, np.zeros(NS), np.zeros(NS))
    if sc_t is not None:
        import torch
        ds.sc_t = torch.stack([torch.from_numpy(np.ascontiguousarray(np.asarray(x).ravel(order="F")))
                               for x in sc_t]).to(ds.dev)
        ds.args.sc_t = ds.sc_t.data_ptr()
    rc = ds.qssa(itchim)
    st = abi.stats()
    tend = ds.tendency_host()
    same_p = all(np.array_equal(a, b) for a, b in zip(ds.species_host(), wl["sc_p"]))
    del ds
    return tend, rc, st, same_p


def _interior(grid):
    return (slice(1, grid.m1 - 1), slice(grid.ia - 1, grid.iz), slice(grid.ja - 1, grid.jz))


def _cell_scale(hs, grid, wl, cells):
    """max(|P/ybid|, |y0|) / conv per species (ppbm) for interior cells
    (j -> i -> k index), from the oracle's gather, kinetic and P/L."""
    lib = O.oracle()
    out = np.zeros((len(cells), NS))
    for n, cell in enumerate(cells):
        y = np.zeros(NS); T = np.zeros(1); p = np.zeros(1); vm = np.zeros(1)
        lib.ora_qssa_gather_cell(O.C.byref(hs.args), int(cell), O.ptr(y), O.ptr(T), O.ptr(p), O.ptr(vm))
        k = 1 + cell % grid.nz
        i = grid.ia - 1 + (cell // grid.nz) % grid.nx
        j = grid.ja - 1 + cell // (grid.nz * grid.nx)
        rk = O.oracle_kinetic(T, p, np.array([float(wl["rv"][k, i, j])]), wl["jphoto"][:, k, i, j][None, :])
        P, L = O.oracle_prod_loss(rk, y[None, :])
        ybid = np.where(L[0] > 0.0, L[0], 1.0)
        conv = np.array([y[s] / float(wl["sc_p"][s][k, i, j]) if wl["sc_p"][s][k, i, j] != 0 else 1.0
                         for s in range(NS)])
        out[n] = np.maximum(np.abs(P[0] / ybid), np.abs(y)) / conv
    return out


def compare(grid, wl, tend_gpu, hs):
    """(worst relative deviation, failures) over every interior cell."""
    idx = _interior(grid)
    dt = float(np.float32(grid.dtlt))
    fails = []
    worst = 0.0
    for s in range(NS):
        old = wl["sc_p"][s][idx].astype(np.float64)
        a = old + tend_gpu[s][idx].astype(np.float64) * dt
        b = old + hs.sc_t[s][idx].astype(np.float64) * dt
        err = np.abs(a - b)
        tol = 1e-6 * np.abs(b) + 1e-7 * np.abs(old) + 1e-30
        worst = max(worst, float(np.max(err / (np.abs(b) + 1e-30))))
        bad = np.nonzero((err > tol).transpose(2, 1, 0).ravel())[0]   # j -> i -> k cell order
        for c in bad:
            fails.append((int(c), s, float(err.transpose(2, 1, 0).ravel()[c])))
    if not fails:
        return worst, 0
    cells = sorted({c for c, _, _ in fails})
    scale = dict(zip(cells, _cell_scale(hs, grid, wl, cells)))
    left = [(c, s, e) for c, s, e in fails if e > 1e-13 * scale[c][s]]
    return worst, len(left)


@pytest.mark.parametrize("seed,sza,plume", [(0, "random", None), (1, "split", None),
                                            (2, "split", 4.0), (3, "split_night_first", 4.0)])
def test_qssa_16x16x10_matches_oracle(seed, sza, plume):
    print("case qssa 16x16x10 seed=%d sza=%s plume=%s" % (seed, sza, plume), flush=True)
    grid = Grid(16, 16, 10)
    wl = make_workload(grid, seed=seed, sza=sza, plume_sigma=plume, all_ppbm=True)
    tend, rc, st, same_p = _gpu(wl)
    hs, orc = O.run_oracle_qssa(wl)
    worst, nfail = compare(grid, wl, tend, hs)
    print("  rc %d/%d, %.3f ms, worst %.3g, beyond bound %d" % (rc, orc, st.kernel_ms, worst, nfail), flush=True)
    assert rc == 0 and orc == 0 and same_p
    assert st.cells == grid.ncell
    assert nfail == 0


def test_qssa_accumulates_into_existing_tendency():
    grid = Grid(9, 7, 6)
    wl = make_workload(grid, seed=5, sza="split", all_ppbm=True)
    rng = np.random.default_rng(1)
    base = [np.asfortranarray(rng.uniform(-1e-3, 1e-3, x.shape).astype(np.float32)) for x in wl["sc_p"]]
    tend, rc, _, _ = _gpu(wl, sc_t=base)
    hs, orc = O.run_oracle_qssa(wl, sc_t=base)
    assert rc == 0 and orc == 0
    _, nfail = compare(grid, wl, tend, hs)
    assert nfail == 0


@pytest.mark.parametrize("nx,ny,nz,itchim", [(1, 1, 1, 1), (9, 7, 1, 2), (8, 4, 2, 3), (13, 5, 1, 64), (5, 13, 3, 75)])
def test_qssa_ragged_groups_match_oracle(nx, ny, nz, itchim):
    """1, 63, 64, 65 and 195 cells, so that the last 64 are partly or wholly
    there, and sub-step counts of one bit, several and all."""
    print("case qssa %dx%dx%d itchim=%d" % (nx, ny, nz, itchim), flush=True)
    grid = Grid(nx, ny, nz)
    wl = make_workload(grid, seed=nx, sza="random", all_ppbm=True)
    base = [np.asfortranarray(np.full_like(x, 0.25)) for x in wl["sc_p"]]
    tend, rc, st, _ = _gpu(wl, itchim, sc_t=base)
    hs, orc = O.run_oracle_qssa(wl, itchim, sc_t=base)
    assert rc == 0 and orc == 0 and st.cells == grid.ncell
    idx = _interior(grid)
    for s in range(NS):
        frame = np.ones(tend[s].shape, bool)
        frame[idx] = False
        assert np.array_equal(tend[s][frame], base[s][frame])
    _, nfail = compare(grid, wl, tend, hs)
    assert nfail == 0


def test_qssa_host_entry_matches_device_entry():
    from brams_amd.chem import run_workload_qssa_host
    grid = Grid(12, 9, 7)
    wl = make_workload(grid, seed=3, all_ppbm=True)
    host, rc = run_workload_qssa_host(wl)
    tend, rc2, _, _ = _gpu(wl)
    assert rc == 0 and rc2 == 0
    for a, b in zip(host, tend):
        assert np.array_equal(a, b)


def test_qssa_host_entry_above_the_staging_size_matches_device_entry():
    """40x40x40: 39 MB of arrays, each copied by itself."""
    from brams_amd.chem import run_workload_qssa_host
    grid = Grid(40, 40, 40)
    wl = make_workload(grid, seed=4, all_ppbm=True)
    host, rc = run_workload_qssa_host(wl)
    tend, rc2, _, _ = _gpu(wl)
    assert rc == 0 and rc2 == 0
    for a, b in zip(host, tend):
        assert np.array_equal(a, b)


def test_qssa_cell_reaching_1e20_is_counted_and_keeps_its_tendency():
    print("case qssa 1e20 cell, 5x4x3", flush=True)
    grid = Grid(5, 4, 3)
    wl = make_workload(grid, seed=8, all_ppbm=True)
    wl["sc_p"][0] = wl["sc_p"][0].copy()
    k, i, j = 2, grid.ia, grid.ja
    wl["sc_p"][0][k - 1, i - 1, j - 1] = 1.0e25
    base = [np.full_like(x, 0.125) for x in wl["sc_p"]]
    tend, rc, st, _ = _gpu(wl, sc_t=base)
    hs, orc = O.run_oracle_qssa(wl, sc_t=base)
    assert rc == orc == 1 and st.failed_blocks == 1
    for s in range(NS):
        assert tend[s][k - 1, i - 1, j - 1] == np.float32(0.125)
    _, nfail = compare(grid, wl, tend, hs)
    assert nfail == 0


def test_qssa_200x200x40_matches_oracle():
    print("case qssa 200x200x40 split plume", flush=True)
    grid = Grid(200, 200, 40, dtlt=120.0)
    wl = make_workload(grid, seed=0, sza="split", plume_sigma=20.0, all_ppbm=True)
    tend, rc, st, same_p = _gpu(wl)
    hs, orc = O.run_oracle_qssa(wl)
    worst, nfail = compare(grid, wl, tend, hs)
    print("  rc %d/%d, %.3f ms, worst %.3g, beyond bound %d" % (rc, orc, st.kernel_ms, worst, nfail), flush=True)
    assert rc == 0 and orc == 0 and same_p
    assert nfail == 0
