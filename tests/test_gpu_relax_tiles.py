"""Tile sizes of the single-scan relaxation (launch_single, relax_dev.hip): a
scan of any size, in tiles of 4 to 64 columns with and without waiting lanes,
gives the bits of the batch kernel, whose tiles have 64 columns.  Sizes: one
column, ragged ones, and on 256 CUs and 1,024 SIMDs the last of 4, 8, 16 and 32
columns a wave (32x32, 64x32, 128x128, 256x128) and one row more."""

import numpy as np
import pytest

from ppafm_amd import batch as B
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
