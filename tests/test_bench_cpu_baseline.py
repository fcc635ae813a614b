"""The benchmark's CPU baseline stays bounded where the reference's build is
absent: the oracle port, whose direct pressure solve costs the fourth power of
the window, gets a smaller one and a time limit."""
import subprocess

import pytest

import bench
import oracle as O


@pytest.fixture
def no_reference(monkeypatch, tmp_path):
    monkeypatch.setattr(O, "REF_BIN", tmp_path / "absent")


def test_port_takes_a_smaller_window(no_reference):
    r = bench.cpu_baseline(bench.workload(64, 3, 1e-8), 48, 1, port_window=12)
    assert r["kind"] == "port" and "12x12x3" in r["sample"]
    assert r["value"] == pytest.approx(12 * 12 * 3 * 2 / r["wall_s"])
    assert bench.PORT_WINDOW <= 32


def test_port_is_stopped_at_its_limit(no_reference):
    with pytest.raises(subprocess.TimeoutExpired):
        bench.cpu_baseline(bench.workload(160, 10, 1e-10), 128, 10, timeout=3.0, port_window=128)
