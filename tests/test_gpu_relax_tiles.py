"""Tile sizes of the single-scan relaxation (launch_single, relax_dev.hip): a
scan of any size, in tiles of 4 to 64 columns with and without waiting lanes,
gives the bits of the batch kernel, whose tiles have 64 columns.  Sizes: one
column, ragged ones, and on 256 CUs and 1,024 SIMDs the last of 4, 8, 16 and 32
columns a wave (32x32, 64x32, 128x128, 256x128) and one row more, and the first scan with
more 64-column tiles than SIMDs (264x257)."""

import numpy as np
import pytest

from ppafm_amd import batch as B
from ppafm_amd import common as C
from ppafm_amd import device as D
from ppafm_amd import molgen as M
from ppafm_amd.scan import PlainScan

pytestmark = pytest.mark.gpu

TIP = dict(tipR0=M.TIP_R0, k_lat=M.K_LAT, k_rad=M.K_RAD, iZPP=M.PROBE_Z, probe_q=M.PROBE_Q, amplitude=M.DF_AMPLITUDE)
LVEC = np.array([[-3.2, -3.2, -3.0], [6.4, 0, 0], [0, 6.4, 0], [0, 0, 12.0]])
N = (64, 64, 120)


@pytest.mark.parametrize("nx,ny", [(1, 1), (3, 5), (32, 32), (33, 32), (64, 32), (65, 32), (64, 64), (70, 70), (91, 90), (128, 128), (129, 128), (181, 181), (256, 128), (256, 129)])
def test_single_scan_equals_batch(nx, ny):
    print(f"case: {nx} x {ny} columns", flush=True)
    scan = dict(scan_n=(nx, ny), scan_x=(-2.5, 2.5), scan_y=(-2.5, 2.5), z_top=6.2, nz=3, dz=0.1)
    mol = M.molecule(18, 5)
    s = PlainScan(LVEC, N, scan, **dict(TIP, amplitude=0.2))
    s.set_molecule(*mol)
    s.run()
    D.synchronize()
    b = B.BatchScan.plain([LVEC], [N], [scan], molecules=[mol], keep_iters=True, **dict(TIP, amplitude=0.2))
    b.run()
    b.synchronize()
    assert np.array_equal(b.positions_raw(0), s.pos.download())
    assert np.array_equal(b.forces(0), s.forces())
    assert np.array_equal(b.iterations(0), s.iterations())
    it = s.iterations().astype(np.int64)
    capped = it >= b.rp.max_iters
    # evaluations: a move each (one more than the recorded count where the stop rule ended the step) and the output sample
    assert int(s.counters.download()[0]) == int(np.where(capped, it, it + 1).sum() + it.size) == b.counters()[0]
    assert int(s.counters.download()[1]) == it.size
    assert 0 < b.lane_use() <= 1
    b.close()


def _many_tiles(f64):
    scan = dict(scan_n=(264, 257), scan_x=(-2.5, 2.5), scan_y=(-2.5, 2.5), z_top=6.2, nz=2, dz=0.1)
    mol = M.molecule(18, 5)
    tip = dict(TIP, amplitude=0.1)
    s = PlainScan(LVEC, N, scan, grid_f64=f64, fp64_radius=0.0, **tip)
    s.set_molecule(*mol)
    s.run()
    D.synchronize()
    b = B.BatchScan.plain([LVEC], [N], [scan], molecules=[mol], keep_iters=True, grid_f64=f64, fp64_radius=0.0, **tip)
    return s, b


@pytest.mark.parametrize("f64", [True, False], ids=["double4", "float4"])
def test_more_tiles_than_simds(f64):
    print("case: 264 x 257 columns", f64, flush=True)
    s, b = _many_tiles(f64)
    b.run()
    b.synchronize()
    assert np.array_equal(b.grid(0), s.grid_host())
    assert np.array_equal(b.positions_raw(0), s.pos.download())
    assert np.array_equal(b.forces(0), s.forces())
    assert np.array_equal(b.iterations(0), s.iterations())
    b.close()


@pytest.mark.parametrize("shear", [0.0, 0.7], ids=["orthogonal", "sheared"])
@pytest.mark.parametrize("f64", [False, True], ids=["float4", "double4"])
@pytest.mark.parametrize("nx,ny", [(1, 1), (33, 32), (65, 32), (129, 128), (256, 129), (264, 257)])
def test_tilted_single_scan_equals_batch(nx, ny, f64, shear):
    """OpenCL semantics (mode 1): another share of waiting lanes, the energy as
    a fourth component, the tip frame's rotation."""
    print(f"case: {nx} x {ny} columns, f64 {f64}, shear {shear}", flush=True)
    lvec = LVEC.copy()
    lvec[1, 1] = shear
    a = 0.2
    rot = np.array([[np.cos(a), 0, np.sin(a)], [0, 1, 0], [-np.sin(a), 0, np.cos(a)]])
    b = B.BatchScan.tilted([lvec], [N], rot=rot, pos0s=[(0.0, 0.0, 6.4)], start=(-2.5, -2.5), end=(2.5, 2.5), scan_n=(nx, ny), nz=11,
                           molecules=[M.molecule(18, 5)], grid_f64=f64, keep_iters=True)
    b.run()
    b.synchronize()
    xyz, Zs, qs = M.molecule(18, 5)
    cLJs = C.REA2LJ(C.getAtomsREA(8, Zs, C.loadSpecies(), alphaFac=-1.0))
    grid = D.ff_build(N, lvec[1:], np.concatenate([xyz - lvec[0], qs[:, None]], 1), cLJs, b.model, f64=f64)
    pos, force, iters = D.relax(N, lvec[1:], grid, b.rp, b.tip, b.items[0]["scan"], pos=True, force=True, iters=True)
    D.synchronize()
    assert np.array_equal(b.grid(0), grid.download())
    assert np.array_equal(b.positions_raw(0), pos.download())
    assert np.array_equal(b.forces(0), force.download())
    assert np.array_equal(b.iterations(0), iters.download())
    b.close()
