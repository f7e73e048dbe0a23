"""The statistic by which casts of small batches choose their waves (OctreeFlat::ray_records): the
records that a random ray meets.  One long leaf in a corner of a scene must not reach the line of 2,048
records from which a batch goes out over more waves; a scene whose every ray meets long leaves must."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import dumbray_amd as D
from dumbray_amd import scenes as S

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "dumbray_amd", "csrc")
LINE = 2048


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include"):
        pytest.skip("g++ or the HIP headers not available")
    exe = str(tmp_path_factory.mktemp("ray_records") / "probe")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-pthread", "-I/opt/rocm/include", "-I" + CSRC,
                    "-D__HIP_PLATFORM_AMD__", "-x", "c++", os.path.join(CSRC, "dr_octree_build.hip"),
                    os.path.join(HERE, "cpp", "ray_records_probe.cpp"), "-o", exe], check=True, capture_output=True)
    return exe


def _with_stack(base, n, size):
    """base and n nearly equal triangles in its middle, `size` of the scene large."""
    rng = np.random.default_rng(0)
    lo, hi = S.scene_aabb(base)
    c, s = (lo + hi) / 2, size * (hi - lo).max()
    t = np.concatenate([c + s * np.array(v) for v in ((-.5, -.4, .1), (.5, -.3, -.1), (0, .6, .05))])[None]
    return np.concatenate([base, t + rng.normal(size=(n, 9)) * s * 1e-4]).astype(np.float32)


def _ico():
    return S.icosphere_scene(4, seed=1).tris


CASES = {
    "mesh": (_ico, False, 100),
    "long leaf out of the way": (lambda: _with_stack(_ico(), 8000, 0.02), False, 8000),
    "long leaf in the way": (lambda: _with_stack(_ico(), 30000, 0.3), True, 30000),
    "stack on a quad": (lambda: _with_stack(S.ground_quad(0.0, 1.0), 3000, 0.01), None, 0),
    "few triangles": (lambda: S.ground_quad(0.0, 1.0), False, 2),
}


@pytest.mark.parametrize("name", list(CASES))
def test_records_a_ray_meets(probe, tmp_path, name):
    make, many, longest = CASES[name]
    tris = np.ascontiguousarray(make(), np.float32)
    tris.tofile(tmp_path / "t.bin")
    out = subprocess.run([probe, str(tmp_path / "t.bin"), "16", "12"], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0
    got = float(out.stdout)
    tree = D.Octree(16, 12)
    tree.push(tris)
    tree.build()
    bounds, children, off, _ = tree.export()
    e = np.diff(np.asarray(bounds, np.float64).reshape(-1, 2, 3), axis=1)[:, 0]
    surface = e[:, 0] * e[:, 1] + e[:, 1] * e[:, 2] + e[:, 2] * e[:, 0]
    counts = np.diff(off) * (np.asarray(children) < 0)
    with np.errstate(all="ignore"):
        share = surface / surface[0]
    want = float((counts * np.where(np.isfinite(share), share, 0.0)).sum())
    assert got == pytest.approx(want, rel=1e-9)
    if name != "mesh" and many is not None:
        assert counts.max() >= longest
    if many is not None:
        assert (got >= LINE) == many
