"""Rays whose direction components are finite but so large that their sum is not: the kernels' walk
(dr_group.h, built for the host) finds what the reference walk finds, bit for bit."""
import subprocess

import numpy as np
import pytest

from test_walk_host import SCENES, _rays, probe  # noqa: F401


@pytest.mark.parametrize("name", list(SCENES))
def test_directions_near_the_largest_float(probe, tmp_path, name):  # noqa: F811
    make, split, depth = SCENES[name]
    tris = np.ascontiguousarray(make(), np.float32)
    base = _rays(tris, 200, seed=len(name))[:1000]
    rays = []
    for largest in (1e38, 3e38, float(np.finfo(np.float32).max)):
        r = base.astype(np.float64)
        r[:, 3:] *= largest / np.abs(r[:, 3:]).max(1, keepdims=True)
        rays.append(r.astype(np.float32))
    rays = np.ascontiguousarray(np.concatenate(rays))
    assert np.isfinite(rays).all()
    with np.errstate(over="ignore"):
        assert np.isinf(np.abs(rays[:, 3:]).sum(1, dtype=np.float32)).mean() > 0.3
    tris.tofile(tmp_path / "tris.bin")
    rays.tofile(tmp_path / "rays.bin")
    r = subprocess.run([probe, str(tmp_path / "tris.bin"), str(tmp_path / "rays.bin"), str(split), str(depth)],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr
    assert int(r.stdout.split()[2]) > len(rays) // 100
