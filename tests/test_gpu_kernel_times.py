"""nhw_kernel_stats names the kernels that ran, counts their launches and
charges each with the bytes that its pass has to move."""
import ctypes as C

import pytest

from nhwave_amd import capi
from nhwave_amd import scenario as S
from nhwave_amd.model import Model

pytestmark = pytest.mark.gpu


def table(m, steps):
    """{kernel: (launches, bytes a launch)} of `steps` steps."""
    capi.check(m.lib.nhw_kernel_timing(m.ctx, 1), "nhw_kernel_timing")
    m.step(steps)
    out = {}
    kid = 0
    while True:
        name, n, ms, b = C.c_char_p(), C.c_int64(), C.c_double(), C.c_double()
        if m.lib.nhw_kernel_stats(m.ctx, kid, C.byref(name), C.byref(n), C.byref(ms), C.byref(b)):
            break
        kid += 1
        if n.value:
            assert name.value.decode() not in out
            out[name.value.decode()] = (n.value, b.value)
    return out


SPLIT = {"k_flux_x", "k_flux_y", "k_flux_z", "k_omega_x", "k_omega_y"}
FUSED = {"k_flux_xyz", "k_omega_xy"}


@pytest.mark.parametrize("precision", [capi.NHW_FP64, capi.NHW_MIXED])
@pytest.mark.parametrize("m,n,k,fused", [(70, 60, 6, True), (512, 384, 8, True), (512, 385, 8, False)])
def test_kernels_of_a_step(gpu, m, n, k, fused, precision):
    s = S.random_scenario(7, mglob=m, nglob=n, kglob=k, dry=False, tol=1e-6)
    with Model(s, precision=precision) as a:
        t = table(a, 2)
    assert (set(t) & (SPLIT | FUSED)) == (FUSED if fused else SPLIT)
    assert not {"k_projection", "k_rk_blend", "k_momenta", "k_copy", "k_mg_tail"} & set(t)
    stages = 2 * s.time_order
    w = 8.0 if precision == capi.NHW_FP64 else 4.0
    cells, columns = m * n * k, m * n
    assert t["k_begin"][0] == 2
    assert t["k_p_from_x"] == (stages, 16.0 * cells)
    # before the solve D U, D V, D W are read and U, V, W written; at the end of
    # a stage also P and the step's momenta are read and the momenta written
    launches, moved = t["k_uvw_a"]
    assert launches == 2 * stages
    least = (6 + 12) / 2 * w * cells + 8.0 * cells / 2
    assert least <= moved <= least + 8.0 * 16 * columns
    faces = [x for x in ("k_flux_xyz", "k_flux_x", "k_flux_y", "k_flux_z") if x in t]
    assert all(t[x][0] == stages for x in faces)
    moved = sum(t[x][1] for x in faces)
    # 6 + 6 + 3 fields and Omega read, 4 + 4 + 3 fluxes written; face planes and 2-D fields besides
    least = (15 + 1 + 11) * w * cells
    assert least <= moved <= 1.3 * least


def test_kernels_of_the_other_forms(gpu):
    s = S.random_scenario(7, mglob=200, nglob=1, kglob=3, dry=False, tol=1e-6)
    with Model(s) as a:
        t = table(a, 1)
    assert "k_mg_tail" in t and "k_coarse" not in t
    s = s.with_(viscous=True, bc=(5, 1, 1, 1, 1), non_hydro=False)
    with Model(s) as a:
        t = table(a, 1)
    cells = 200 * 3
    assert t["k_momenta"][0] == s.time_order
    assert 9 * 8.0 * cells <= t["k_momenta"][1] <= 9 * 8.0 * cells + 8.0 * 2 * 200
