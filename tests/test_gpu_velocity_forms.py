"""The forms of the velocity pass at the end of a stage: groups of two levels
(an odd number leaves one of one) and the one group of three, sides that
mirror, inflow, open and wall friction sides, hydrostatic and not, alone and
side by side in a batch.

Against the oracle: hydrostatic, the same operations but for the boundary
signals' and the log law's libm (1e-12 of each field's largest value after three
steps); non-hydrostatic, its direct solve against TOL 1e-12 (1e-9 on the
velocities).  A batch's hydrostatic members are the single runs bit for bit, in
FP64 and in the mixed form."""
from dataclasses import replace

import numpy as np
import pytest

import oracle as O
from nhwave_amd import capi
from nhwave_amd import scenario as S
from nhwave_amd.batch import Batch
from nhwave_amd.model import Model

pytestmark = pytest.mark.gpu
FIELDS = ("Eta", "U", "V", "W", "DU", "DV", "DW")


def case(sides, k, non_hydro):
    if sides == "inflow":
        s = S.wave_flume(mglob=40, nglob=5, kglob=k, dx=0.05, wavemaker="LEF_LIN", amp=0.02, per=1.0, theta=10.0,
                         bottom="bar", tol=1e-12)
    elif sides == "open":
        s = S.steady_flume(mglob=40, nglob=4, kglob=k, dx=0.05, obstacle=0.05, tramp=1.0, zob=1e-3, tol=1e-12)
    else:
        s = S.random_scenario(11, mglob=31, nglob=9, kglob=k, dry=sides == "walls", tol=1e-12)
        if sides == "noslip":
            s = replace(s, bc=(2, 2, 2, 2, 1))
        if sides == "friction":
            s = replace(s, bc=(5, 1, 2, 5, 1), viscous=True, visc=1.0e-3)
    return replace(s, non_hydro=non_hydro)


@pytest.mark.parametrize("non_hydro", [False, True])
@pytest.mark.parametrize("k", [2, 3, 4, 5])
@pytest.mark.parametrize("sides", ["walls", "noslip", "inflow", "open", "friction"])
def test_form_vs_oracle(gpu, sides, k, non_hydro):
    s = case(sides, k, non_hydro)
    o = O.Oracle(s)
    o.step(3)
    with Model(s) as m:
        m.step(3)
        got = m.download(*FIELDS)
    for q in FIELDS:
        inner = (slice(2, -2),) * got[q].ndim
        a, b = got[q][inner], np.asarray(o.field(q))[inner]
        top = max(float(np.abs(np.asarray(o.field("U" if q in "UVW" else "DU" if q != "Eta" else q))).max()), 1e-300)
        assert float(np.abs(a - b).max()) <= (1e-9 if non_hydro else 1e-12) * top, q


@pytest.mark.parametrize("precision", [capi.NHW_FP64, capi.NHW_MIXED])
@pytest.mark.parametrize("sides", [("walls", "noslip", "inflow"), ("walls", "inflow", "friction")])
def test_forms_side_by_side(gpu, sides, precision):
    sc = [case(q, k, False) for k in (2, 3, 4, 5) for q in sides]
    with Batch(sc, precision=precision, autotune=False) as b:
        b.step(3)
        got = [m.download(*FIELDS) for m in b.members]
    for s, g in zip(sc, got):
        with Model(s, precision=precision) as m:
            m.step(3)
            ref = m.download(*FIELDS)
        assert [q for q in FIELDS if not np.array_equal(g[q], ref[q], equal_nan=True)] == [], s.name
