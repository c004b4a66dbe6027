"""The substep kernel with several levels per thread (shape 13) at the edges of its ranges: one and two columns beyond a
block, 63, 64, 127 and 128 levels (where the block widths and the form of the column recurrences change), the smallest
periodic grid, mirrored and open sides, an x-z slice.  Every form of the kernel keeps one order of operations, so its
results are the bits of the level-per-thread shape, in FP64 (which the oracle pins, here too) and in FP32-bulk."""
import numpy as np
import pytest

from cppwrf_amd import _abi as A
from cppwrf_amd.dyn import Case, Context, RK3
from oracle_lib import OracleDomain

pytestmark = pytest.mark.gpu

STATE = (A.MI_U, A.MI_V, A.MI_W, A.MI_T, A.MI_PH, A.MI_MU, A.MI_P, A.MI_AL)
P, S, O = A.MI_BC_PERIODIC, A.MI_BC_SYMMETRIC, A.MI_BC_OPEN
GRIDS = [(3, 3, 5, P), (9, 5, 62, P), (10, 4, 63, P), (7, 8, 64, O), (8, 4, 127, S), (17, 5, 128, P), (5, 3, 200, P), (66, 1, 20, S)]


@pytest.fixture(scope="module")
def ctx():
    return Context(0)


@pytest.mark.parametrize("nx,ny,nz,bc", GRIDS)
@pytest.mark.parametrize("precision", [A.MI_FP64, A.MI_FP32_BULK])
def test_levels_per_thread_bits(ctx, nx, ny, nz, bc, precision):
    print(f"[levels] {nx}x{ny}x{nz} bc {bc} precision {precision}", flush=True)
    case = Case.bubble3d(nx, ny, nz, dx=1000.0, ztop=min(200.0 * nz, 20000.0), dt=2.0, seed=nx + nz, noise_amp=0.3, bubble_zc=min(40.0 * nz, 4000.0), bc=bc)
    kw = dict(time_step_sound=4, damp_opt=3, zdamp=min(60.0 * nz, 6000.0), top_lid=1 if nz == 64 else 0)
    per_thread = 4 if nz + 1 <= 64 else (5 if nz + 1 <= 128 else 6)
    doms = []
    for shape in (per_thread, 13):
        d = RK3(ctx, case.grid, case.params(precision=precision, **kw), case)
        t = d.tuning
        t[2] = shape
        d.tuning = t
        d.step(2)
        assert d.check_finite() == -1
        doms.append(d)
    for fid in STATE:
        x, y = (d.field(fid) for d in doms)
        assert np.array_equal(x.view(np.uint64), y.view(np.uint64)), A.FIELD_NAMES[fid]
    if precision == A.MI_FP64:
        orc = OracleDomain(case, case.params(**kw))
        orc.step(2)
        for fid in STATE:
            assert np.array_equal(doms[1].field(fid).view(np.uint64), orc.field(fid).view(np.uint64)), A.FIELD_NAMES[fid]
