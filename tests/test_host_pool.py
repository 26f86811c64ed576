"""The host threads of large loads and readbacks: the pool by itself (tests/cpp/pool_check.cpp,
CPU), and records that pass through it unchanged (GPU)."""

import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_item_once(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    exe = str(tmp_path / "pool_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "pool_check.cpp"),
                    os.path.join(ROOT, "cellflow_amd", "csrc", "cf_host.cpp")], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and "pool ok" in out.stdout, (out.returncode, out.stderr)


# around the sizes where a load is staged, sliced and shared (44-byte records; 128 KiB per
# range, 2 MiB per slice, 16 slices at most)
@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2978, 8935, 47662, 47663, 95325, 95326, 400000, 800009])
def test_records_round_trip(n):
    from cellflow_amd import CellFlowError, ParticleSimulation
    from cellflow_amd.simulation import PARTICLE_DTYPE
    rng = np.random.default_rng(n)
    rec = np.zeros(n, PARTICLE_DTYPE)
    for f in ("pos", "vel", "acc"):
        rec[f] = rng.random((n, 3), np.float32)
    rec["ptype"] = rng.integers(0, 5, n)
    rec["pad"] = rng.random(n, np.float32)
    with ParticleSimulation(n, 5) as sim:
        for _ in range(2):  # before and after the staging buffer exists
            sim.setParticles(rec)
            out = np.zeros_like(rec)
            assert sim.getParticleData(out=out).tobytes() == rec.tobytes()
            # one bad type anywhere: refused, named, and nothing changed
            for at in {0, n // 2, n - 1}:
                bad = rec.copy()
                bad["pos"] += 1
                bad["ptype"][at] = 5
                with pytest.raises(CellFlowError, match=f"particle {at} has type 5"):
                    sim.setParticles(bad)
            assert sim.getParticleData().tobytes() == rec.tobytes()
            rec["pos"] *= np.float32(0.5)
