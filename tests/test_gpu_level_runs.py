"""Options and boundaries with runs of several levels per thread (grids with enough wavefronts per level), two steps.

FP64: every prognostic field, species and forcing has the oracle's bits.

FP32-bulk: the change of every field over the two steps is within 5 % (relative L2) of FP64's.  Storage rounds a value
by 6e-8 of it about ten times in two steps; the fields change by 1e-5 of their size or more in them, so rounding makes
up to 2 % of the change, while a flux missing or misplaced at the seams of runs of 2 to 6 levels makes tens of per
cent."""
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT, bitwise_equal, first_diff
from cppwrf_amd import _abi as A
from cppwrf_amd.boundary import drifting_boundary
from cppwrf_amd.dyn import Case, Context, RK3
from cppwrf_amd.workloads import moist_species, rel_l2
from oracle_lib import OracleDomain
from physics_plugin import Plugin

pytestmark = pytest.mark.gpu

STATE = (A.MI_U, A.MI_V, A.MI_W, A.MI_T, A.MI_PH, A.MI_MU, A.MI_P, A.MI_AL)
P, O, B = A.MI_BC_PERIODIC, A.MI_BC_OPEN, A.MI_BC_SPECIFIED


def _hills(bc, seed, nz=20):
    return lambda: Case.hills(198, 121, nz, dx=15000.0, dt=60.0, seed=seed, bc=bc)


def _bubble(nx, ny, nz, bc, **kw):
    return lambda: Case.bubble3d(nx, ny, nz, seed=nz, noise_amp=0.3, bc=bc, bubble_zc=3000.0, **kw)


CASES = {  # name: (case, parameters, the plugin's forcings kept)
    # the vapour stores RQVFTEN, level by level, beside species whose runs march: plain and limited, in one list or two
    "forcing_periodic": (_hills(P, 3), dict(n_moist=2, n_scalars=4, moist_adv_opt=1, scalar_adv_opt=0), True),
    "forcing_specified": (_hills(B, 4), dict(n_moist=3, n_scalars=3, moist_adv_opt=1), True),
    "forcing_plain": (_hills(P, 5), dict(n_moist=1, n_scalars=1, moist_adv_opt=0), True),
    "forcing_tracer_limited": (_hills(P, 6), dict(n_moist=1, n_scalars=2, moist_adv_opt=0, scalar_adv_opt=1), True),
    # open sides: advance_uv, small_step_prep, calc_cq and the limiter's scale take runs there too
    "open_limited": (_hills(O, 9), dict(n_moist=3, n_scalars=4, moist_adv_opt=1, scalar_adv_opt=1), False),
    "open_dry": (_bubble(257, 190, 33, O, dx=3000.0, ztop=16000.0, dt=10.0), {}, False),
    # the rigid lid, and updraughts beyond a vertical Courant number of 1 (set below) that w_damping pulls back
    "lid_w_damping": (_bubble(198, 149, 24, P, dx=10000.0, ztop=8000.0, dt=20.0),
                      dict(time_step_sound=8, top_lid=1, w_damping=1, zdamp=2000.0), False),
    "specified_six": (_hills(B, 10, 23), dict(n_moist=6, n_scalars=6, moist_adv_opt=1, diff_6th_opt=1), False),
    "lid_tall": (_bubble(130, 129, 70, P, dx=1000.0, ztop=18000.0, dt=2.0), dict(top_lid=1), False),
}


@pytest.fixture(scope="module")
def ctx():
    return Context(0)


@pytest.mark.parametrize("name", list(CASES))
def test_runs_of_levels(ctx, name):
    print(f"[level runs] {name}", flush=True)
    make, opts, forcing = CASES[name]
    case = make()
    kw = dict(dict(time_step_sound=4, damp_opt=3, zdamp=5000.0), **opts)
    ns = kw.get("n_scalars", 0)
    doms = [RK3(ctx, case.grid, case.params(precision=p, **kw), case) for p in (A.MI_FP64, A.MI_FP32_BULK)]
    orc = OracleDomain(case, case.params(**kw))
    fids = STATE + tuple(A.MI_Q + n for n in range(ns))
    for d in doms + [orc]:
        if case.grid.bc_x == B:
            d.load_boundary(drifting_boundary(case, seed=5))
        for fid, q in (moist_species(case, ns, seed=7) if ns else {}).items():
            d.set_field(fid, q)
        if kw.get("w_damping"):
            z, _, x = np.indices(A.field_shape(A.MI_U, case.grid.nx, case.grid.ny, case.grid.nz))
            d.set_field(A.MI_U, 180.0 * np.sin(2 * np.pi * x / 11) * (z < case.grid.nz // 2))
        if forcing:
            d.set_column_physics(Plugin(True, True, ns))
    before = [{f: d.field(f) for f in fids} for d in doms]
    for d in doms + [orc]:
        d.step(1)
        assert not kw.get("w_damping") or d.cfl_max()[0] > 1.0
        d.step(1)
    for fid in fids + ((A.MI_TH_FORCING, A.MI_QV_FORCING) if forcing else ()):
        a, b = doms[0].field(fid), orc.field(fid)
        assert bitwise_equal(a, b), f"{A.FIELD_NAMES[fid]}: {first_diff(a, b)}"
    for fid in fids:
        change = [d.field(fid) - b[fid] for d, b in zip(doms, before)]
        e = rel_l2(change[1], change[0])
        print(f"[level runs] {name} {A.FIELD_NAMES[fid]}: {e:.2e}", flush=True)
        assert e <= 5e-2, A.FIELD_NAMES[fid]


_STEP = """
import sys
import numpy as np
from cppwrf_amd import _abi as A
from cppwrf_amd.dyn import Case, Context, RK3
ctx = Context(0)
for p in (A.MI_FP64, A.MI_FP32_BULK):
    case = Case.hills(198, 121, 20, dx=15000.0, dt=60.0, seed=8)
    d = RK3(ctx, case.grid, case.params(precision=p, time_step_sound=4, damp_opt=3, n_moist=2, n_scalars=2), case)
    d.step(2)
    np.save(f"{sys.argv[1]}_{p}.npy", np.concatenate([d.field(f).ravel() for f in case.STATE + (A.MI_Q, A.MI_Q + 1)]))
"""


def test_block_order_keeps_the_bits(ctx, tmp_path):
    """MI_BLOCK_ORDER=ijk (read once per process) gives every point kernel's blocks, runs of levels included, the i, j,
    level order: the same results"""
    for order in ("", "ijk"):
        print(f"[level runs] block order {order!r}", flush=True)
        subprocess.run([sys.executable, "-c", _STEP, str(tmp_path / ("o" + order))], check=True, cwd=ROOT, timeout=100,
                       env=dict(os.environ, MI_BLOCK_ORDER=order))
    for p in (A.MI_FP64, A.MI_FP32_BULK):
        a, b = (np.load(tmp_path / f"o{o}_{p}.npy") for o in ("", "ijk"))
        assert bitwise_equal(a, b), p
