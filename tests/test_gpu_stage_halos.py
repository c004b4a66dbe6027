"""The halos a caller sees through a field's view after each phase of the phase-by-phase step (the reference refreshes them
there, small_step.cpp:517-606): every halo point of the stage's mass fields holds the value of the point its boundary
condition names, corners included."""
import ctypes as C

import numpy as np
import pytest

from cppwrf_amd import _abi as A
from cppwrf_amd.dyn import Case, Context, RK3

pytestmark = pytest.mark.gpu

P, S, O, B = A.MI_BC_PERIODIC, A.MI_BC_SYMMETRIC, A.MI_BC_OPEN, A.MI_BC_SPECIFIED
NH = 3


@pytest.fixture(scope="module")
def ctx():
    return Context(0)


def _with_halo(d, fid):
    """the field's storage through its view, halos included: (nz, ny + 2 hy, nx + 6)"""
    v = d.field_view(fid)
    e, hy = v.elem_bytes, NH if v.stride_j else 0
    first = -(hy * v.stride_j + NH)
    n = (v.ny - 1 + hy) * v.stride_j + (v.nz - 1) * v.stride_k + v.nx + NH - first
    buf = np.empty(n, dtype=np.float64 if e == 8 else np.float32)
    hip = C.CDLL("libamdhip64.so")
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    d.sync()
    assert hip.hipMemcpy(buf.ctypes.data, v.data + first * e, buf.nbytes, 2) == 0
    k, j, i = np.meshgrid(np.arange(v.nz), np.arange(-hy, v.ny + hy), np.arange(-NH, v.nx + NH), indexing="ij")
    return buf[i + k * v.stride_k + j * v.stride_j - first], hy


def _source(n, bc, halo):
    i = np.arange(-halo, n + halo)
    if bc == P:
        return i % n
    if bc == S:
        return np.where(i < 0, -1 - i, np.where(i >= n, 2 * n - 1 - i, i))
    return np.clip(i, 0, n - 1)


@pytest.mark.parametrize("precision", [A.MI_FP64, A.MI_FP32_BULK])
@pytest.mark.parametrize("nx,ny,bc,bc_y", [(20, 16, P, P), (17, 12, S, P), (18, 15, O, S), (24, 1, P, P)])
def test_halos_after_the_small_steps(ctx, nx, ny, bc, bc_y, precision):
    print(f"[stage halos] {nx}x{ny} bc {bc} {bc_y} precision {precision}", flush=True)
    case = Case.bubble3d(nx, ny, 12, dx=1000.0, ztop=8000.0, dt=6.0, seed=4, noise_amp=0.3, bc=bc, bc_y=bc_y)
    d = RK3(ctx, case.grid, case.params(precision=precision, time_step_sound=4, damp_opt=3, zdamp=3000.0), case)
    d.step_begin()
    for rk in (1, 2, 3):
        d.rk_prep(rk)
        d.rk_tendency(rk)
        d.small_steps(rk)
        for fid in (A.MI_P, A.MI_AL, A.MI_PH, A.MI_T, A.MI_W, A.MI_MU, A.MI_MUTS, A.MI_WW, A.MI_WW_M):
            got, hy = _with_halo(d, fid)
            inner = got[:, hy:hy + ny, NH:NH + nx]
            assert np.abs(inner).max() > 0
            want = inner[:, _source(ny, bc_y, hy)][:, :, _source(nx, bc, NH)]
            assert np.array_equal(got, want), f"stage {rk}: {A.FIELD_NAMES[fid]}"
        d.scalar_transport(rk)
        d.calc_p_rho_phi(rk)
