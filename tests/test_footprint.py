"""nhw_footprint gives the device bytes that nhw_create allocates, to the byte:
a serving loop admits requests by it.  The library runs in a child process
whose HIP allocation calls are stood in for (count_device_bytes.c), so no GPU
is needed."""
import json
import os
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CHILD = """
import ctypes as C, json, sys
from nhwave_amd import capi
from nhwave_amd.model import make_config
from nhwave_amd import scenario as S
lib = capi.load()
seen = C.CDLL(sys.argv[1])
seen.counted_bytes.restype = C.c_longlong
seen.counted_of_size.argtypes = [C.c_longlong]
out = []
for c in json.loads(sys.argv[2]):
    m, n, k = c["size"]
    s = S.Scenario(name="", mglob=m, nglob=n, kglob=k, dx=1.0, dy=1.0, hcg=None, etag=None, **c.get("fields", {}))
    cfg = make_config(s, precision=c.get("precision", 0), solver=c.get("solver", 0))
    want = C.c_int64()
    capi.check(lib.nhw_footprint(C.byref(cfg), C.byref(want)), "nhw_footprint")
    seen.counted_clear()
    ctx = C.c_void_p()
    capi.check(lib.nhw_create(C.byref(cfg), C.byref(ctx)), "nhw_create")
    rows = m * n * k * (4 if c.get("precision", 0) else 8)
    out.append([want.value, seen.counted_bytes(), seen.counted_of_size(rows)])
    lib.nhw_destroy(ctx)
print(json.dumps(out))
"""


@pytest.fixture(scope="module")
def created(tmp_path_factory):
    """[footprint, bytes allocated, allocations of one solver vector] of each
    configuration."""
    so = tmp_path_factory.mktemp("count") / "count_device_bytes.so"
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(so), str(ROOT / "tests" / "count_device_bytes.c")], check=True)

    def run(configs):
        env = dict(os.environ, PYTHONPATH=str(ROOT))
        env["LD_PRELOAD"] = " ".join(filter(None, [str(so), env.get("LD_PRELOAD")]))
        r = subprocess.run([sys.executable, "-c", CHILD, str(so), json.dumps(configs)], env=env, cwd=ROOT,
                           capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr
        return json.loads(r.stdout.splitlines()[-1])

    return run


# grids of one multigrid level and of several, of at most 131072 rows and of more, narrow and wide
SIZES = [(12, 12, 3), (32, 32, 16), (70, 1, 4), (83, 41, 6), (128, 64, 16), (129, 64, 16), (256, 128, 4), (2, 20000, 8),
         (1024, 1024, 10)]
SOLVERS = [dict(), dict(precision=1), dict(solver=1)]


def test_footprint_is_what_is_allocated(created):
    configs = [dict(size=z, **q) for z in SIZES for q in SOLVERS]
    configs.append(dict(size=(30, 20, 200), solver=1))
    for z in ((40, 30, 5), (300, 200, 8)):
        configs += [dict(size=z, fields=f) for f in (
            dict(non_hydro=False), dict(sponge=(1.0, 0.0, 0.0, 0.0)), dict(viscous=True), dict(viscous=True, turb=10),
            dict(wavemaker="LEF_LIN", bc=(3, 1, 1, 1, 1), amp_wave=0.1, per_wave=2.0, dep_wave=1.0),
            dict(wavemaker="LEF_SOL", bc=(3, 1, 1, 1, 1), amp_wave=0.1, dep_wave=1.0),
            dict(wavemaker="INT_IRR", dep_wave=1.0), dict(wavemaker="FLUX_LR", bc=(3, 3, 1, 1, 1), zob=1e-3))]
        configs.append(dict(size=z, fields=dict(non_hydro=False), precision=1))
    wrong = [(c, want, got) for c, (want, got, _) in zip(configs, created(configs)) if want != got]
    assert wrong == []


def test_second_direction_only_where_it_is_used(created):
    """The multigrid solver keeps two copies of its direction where the cycle
    forms it as it reads it: solves of several levels and at most 131072 rows.
    Vectors of one number a row: rhs, r, rh, p, v, s, t (mixed: e, r, rh, p, v,
    s, t, ph, sh) and the second p."""
    two = {(12, 12, 3): 0, (32, 32, 16): 0, (70, 1, 4): 1, (83, 41, 6): 1, (128, 64, 16): 1, (129, 64, 16): 0,
           (256, 128, 4): 1, (2, 20000, 8): 0, (1024, 1024, 10): 0}
    assert sorted(two) == sorted(SIZES)
    configs = [dict(size=z, precision=p) for z in SIZES for p in (0, 1)]
    for c, (_, _, vectors) in zip(configs, created(configs)):
        assert vectors == (9 if c["precision"] else 7) + two[tuple(c["size"])], c
