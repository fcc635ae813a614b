"""The velocity pass's U = DU / D over the whole range of momenta: the quotient
that IEEE division gives, to the bit, but for momenta below 2^-900, which may
come out one unit off.  Overflow gives infinity, which the time step
estimate reports; NaN it would pass over."""
import numpy as np
import pytest

from nhwave_amd import capi
from nhwave_amd import scenario as S
from nhwave_amd.model import Model

pytestmark = pytest.mark.gpu
G = S.NGHOST
IN3 = (slice(G, -G),) * 3
BIG = float(np.finfo(np.float64).max)
SPECIAL = [0.0, np.inf, -np.inf, np.nan, BIG, -BIG, BIG / 2, 1e308, -1e300, 2.0**-1022, -2.0**-1022, 5e-324, 3e-320,
           2.0**-1060, 1e-300, 2.0**-900, 1.0, -3.0, 1.0 / 3.0]


def basin(m=65, n=17, k=5):
    rng = np.random.default_rng(3)
    h = 10.0 ** rng.uniform(-1.5, 4.0, (n, m))
    return S.Scenario(name="basin", mglob=m, nglob=n, kglob=k, dx=1.0, dy=1.0, hcg=h, etag=np.zeros((n, m)),
                      non_hydro=False, froude_cap_on=False)


def end_of_stage(m, du):
    """eval_duvw on momenta `du` and face fluxes of zero: DU, D and U after it"""
    f = m.field("DU")
    f[IN3] = du
    m.upload({"DU": f})
    m.call("nhw_eval_duvw", 1)
    got = m.download("DU", "D", "U")
    return got["DU"][IN3], got["D"][G:-G, G:-G], got["U"][IN3]


@pytest.mark.parametrize("precision", [capi.NHW_FP64, capi.NHW_MIXED])
def test_velocities_are_the_quotients(gpu, precision):
    s = basin()
    rng = np.random.default_rng(5)
    shape = (s.kglob, s.nglob, s.mglob)
    lo, hi = (-1074.0, 1024.0) if precision == capi.NHW_FP64 else (-149.0, 127.9)
    x = np.exp2(rng.uniform(lo, hi, shape)) * rng.choice([-1.0, 1.0], shape)
    x.reshape(-1)[:4 * len(SPECIAL):4] = SPECIAL
    x.reshape(-1)[-2000:] = BIG * rng.uniform(0.0, 1.0, 2000)
    if precision == capi.NHW_MIXED:
        with np.errstate(over="ignore"):
            x = x.astype(np.float32).astype(np.float64)
    with Model(s, precision=precision) as m:
        du, d, u = end_of_stage(m, x)
    assert np.array_equal(du, x, equal_nan=True)
    with np.errstate(over="ignore", invalid="ignore", under="ignore"):
        want = x / d[None]
        if precision == capi.NHW_MIXED:
            want = want.astype(np.float32).astype(np.float64)
        small = np.abs(x) < 2.0**-900
        assert np.array_equal(u[~small], want[~small], equal_nan=True)
        assert np.all(np.abs(u[small] - want[small]) <= np.spacing(np.abs(want[small])))


def test_overflowing_velocity_is_reported(gpu):
    s = basin()
    x = np.zeros((s.kglob, s.nglob, s.mglob))
    x[2, 3, 4] = BIG
    s.hcg[3, 4] = 0.5
    with Model(s) as m:
        _, _, u = end_of_stage(m, x)
        assert u[2, 3, 4] == np.inf
        with pytest.raises(capi.NhwError) as e:
            m.call("nhw_estimate_dt")
        assert e.value.code == capi.NHW_EDT
