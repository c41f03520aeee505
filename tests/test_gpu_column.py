"""The acoustic column kernel (k_ac_column) on the GPU (needs an MI355X): one whole step at the
edges of its tile shapes equals the oracle's bit for bit.  The widths put a last tile of one
column, a single tile and whole tiles on a row; the levels sit at and just past what 32-, 16-
and 8-column tiles hold; 321 levels are beyond every tile (the routine kernels)."""
import numpy as np
import pytest

from parity import interior
from wrf_amd import grid, runtime

pytestmark = pytest.mark.gpu

KINDS = dict(u_2="u", v_2="v", w_2="w", t_2="mass", mu_2="mass", p="mass", ph_2="w", al="mass", q0="mass")


@pytest.mark.parametrize("nx,ny,nz,bc,pad", [(33, 12, 48, "periodic", 32), (33, 12, 49, "open", 32), (28, 11, 64, "periodic", 32),
                                             (64, 9, 65, "open", 32), (65, 10, 80, "periodic", 1), (32, 9, 81, "periodic", 32),
                                             (17, 9, 96, "open", 32), (23, 9, 97, "periodic", 32), (15, 9, 161, "periodic", 32),
                                             (18, 9, 193, "open", 1), (9, 8, 320, "periodic", 32), (9, 8, 321, "periodic", 32),
                                             (330, 210, 48, "periodic", 32)])
def test_column_tiles_bitwise(nx, ny, nz, bc, pad):
    import torch
    from pyoracle import Oracle
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a visible GPU")
    print(f"column tiles {nx}x{ny}x{nz} {bc} pad {pad}", flush=True)
    hs = grid.build_initial_state(grid.DomainSpec(nx=nx, ny=ny, nz=nz, bc=bc, n_bubbles=1, seed=nx * nz, pad_i=pad))
    dev = runtime.DeviceDomain(hs)
    dev.step(1)
    got = dev.download()
    exp = Oracle("f32cr").run(hs, 1)
    bad = [k for k, kind in KINDS.items() if not np.array_equal(interior(got[k], hs.dims, kind), interior(exp[k], hs.dims, kind))]
    assert not bad, f"{bad} differ from the oracle"
