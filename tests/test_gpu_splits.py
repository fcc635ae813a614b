"""The splits of the explicit step's sweeps (levels of the x faces, rows of
the y faces, levels of the sigma faces, level groups of the velocity pass) at
sizes around their edges: every persistent array, ghost cells included, equals
the oracle's bit for bit after each of three hydrostatic steps, alone and as
members of one batch (whose sweeps are not split).  One-row grids are compared
in the interior: the second ghost row there mirrors a row that does not exist,
and the device leaves it as it is.

From two levels, a single row and three columns, where each walk is cut to one
step, to 900 x 200 x 12, where none is.  The Froude cap is out of reach: its
cos, sin and atan2 are the device's own."""
from dataclasses import replace

import numpy as np
import pytest

import oracle as O
from nhwave_amd import scenario as S
from nhwave_amd.batch import Batch
from nhwave_amd.model import Model
from test_gpu_parity import FULL

pytestmark = pytest.mark.gpu


def case(m, n, k, bc=(1, 1, 1, 1, 1), order=2):
    return replace(S.random_scenario(5, mglob=m, nglob=n, kglob=k, steps=3, non_hydro=False), bc=bc,
                   time_order=order, froude_cap=1e6)


def differing(s, got, o):
    cut = (slice(2, -2),) if s.nglob == 1 else (slice(None),)
    return [q for q in FULL if not np.array_equal(got[q][cut * got[q].ndim], o.field(q)[cut * got[q].ndim])]


SIZES = [(3, 1, 2), (61, 1, 3), (62, 2, 5), (63, 17, 4), (20, 15, 7), (125, 16, 2), (257, 33, 5), (130, 70, 16)]
WALLS = [(1, 1, 1, 1, 1), (2, 1, 2, 1, 2), (1, 2, 1, 2, 1)]


@pytest.mark.parametrize("m,n,k", SIZES + [(900, 200, 12)])
def test_split_sweeps_vs_oracle(gpu, m, n, k):
    s = case(m, n, k, WALLS[(m + n) % 3], 3 if k == 7 else 2)
    o = O.Oracle(s)
    with Model(s) as a:
        for st in range(3):
            a.step(1)
            o.step(1)
            assert differing(s, a.download(*FULL), o) == [], st


def test_split_sweeps_in_a_batch(gpu):
    members = [case(m, n, k, WALLS[(m + n) % 3]) for m, n, k in SIZES]
    with Batch(members, autotune=False) as b:
        b.step(3)
        for s, a in zip(members, b.members):
            o = O.Oracle(s)
            o.step(3)
            assert differing(s, a.download(*FULL), o) == [], s.name
