"""The traversal's compact child boxes and its deferred slab tests (dr_group.h), built for the host:
the walk that the kernels make finds the reference walk's triangle and distance, bit for bit, for
every form of ray, on trees whose boxes nest and on trees whose boxes do not."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from dumbray_amd import scenes as S

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "dumbray_amd", "csrc")


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include"):
        pytest.skip("g++ or the HIP headers not available")
    exe = str(tmp_path_factory.mktemp("walk_probe") / "walk_probe")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-pthread", "-I/opt/rocm/include", "-I" + CSRC,
                    "-D__HIP_PLATFORM_AMD__", "-x", "c++", os.path.join(CSRC, "dr_octree_build.hip"),
                    os.path.join(HERE, "cpp", "walk_probe.cpp"), "-o", exe], check=True, capture_output=True)
    return exe


def _rays(tris, n, seed):
    """Uniform rays, rays at centroids and vertices from near and far, axis-parallel rays (some with
    an origin on a box plane), rays in a coordinate plane, short and long directions, and rays that
    cannot hit (zero, infinite, NaN)."""
    rng = np.random.default_rng(seed)
    lo, hi = S.scene_aabb(tris)
    size = (hi - lo).max() + 1e-6
    pick = lambda k: tris[rng.integers(0, len(tris), k)]
    out = [S.incoherent_rays(tris, n, seed=seed)]
    for spread in (0.6, 50.0):
        t = pick(n).reshape(-1, 3, 3)
        aim = np.where(rng.random((n, 1)) < 0.5, t.mean(1), t[:, 0])
        o = (lo + hi) / 2 + rng.normal(0, spread * size, (n, 3))
        out.append(np.concatenate([o, aim - o], 1))
    p = pick(n)[:, :3] + rng.normal(0, 0.01 * size, (n, 3)) * (rng.random((n, 1)) < 0.7)
    axis = np.eye(3)[rng.integers(0, 3, n)] * np.where(rng.random((n, 1)) < 0.5, 1.0, -1.0)
    out.append(np.concatenate([p - axis * size * rng.random((n, 1)), axis], 1))
    # origins on the planes of the scene's box
    q = p.copy()
    k = rng.integers(0, 3, n)
    q[np.arange(n), k] = np.where(rng.random(n) < 0.5, lo[k], hi[k])
    out.append(np.concatenate([q, np.where(np.arange(3)[None] == k[:, None], 0.0, rng.normal(size=(n, 3)))], 1))
    base = np.concatenate(out).astype(np.float32)
    scaled = base[rng.integers(0, len(base), n)].copy()
    scaled[:, 3:] *= (np.float32(10.0) ** rng.integers(-34, 30, (n, 1))).astype(np.float32)
    flat = base[rng.integers(0, len(base), n)].copy()
    flat[:, 3:] *= (np.float32(10.0) ** rng.integers(-12, 1, (n, 3))).astype(np.float32)
    dead = base[:64].copy()
    dead[np.arange(64), rng.integers(0, 6, 64)] = rng.choice(np.array([np.nan, np.inf, -np.inf], np.float32), 64)
    dead[:8, 3:] = 0.0
    return np.ascontiguousarray(np.concatenate([base, scaled, flat, dead]), np.float32)


SCENES = {
    "soup": (lambda: S.random_soup(1500, seed=1, extent=10.0, size=1.5), 16, 12),
    "heightfield": (lambda: S.heightfield(48, seed=2), 16, 12),
    "icospheres": (lambda: S.icosphere_scene(4, seed=3).tris, 8, 24),
    "spheres": (lambda: S.spheres_scene(8, seed=0).tris, 16, 12),
    # geometry smaller than the splits' overlap: children poke out of their parents
    "tiny": (lambda: S.random_soup(600, seed=4, extent=0.01, size=0.003), 4, 8),
    "far": (lambda: S.random_soup(800, seed=5, extent=3.0, size=0.5) + np.float32(4096.0), 8, 12),
    "huge": (lambda: S.random_soup(800, seed=6, extent=3e6, size=5e5), 8, 12),
    # axis-parallel walls and floors
    "boxes": (lambda: np.concatenate([S.ground_quad(y, 3.0, x, x) for y in (-1.0, 0.0, 0.5) for x in range(-6, 6)]
                                     + [S.ground_quad(y, 3.0, x, x).reshape(-1, 3)[:, [1, 0, 2]].reshape(-1, 9)
                                        for y in (-1.0, 2.0) for x in range(-6, 6)]).astype(np.float32), 4, 12),
}


@pytest.mark.parametrize("name", list(SCENES))
def test_compact_walk_equals_reference_walk(probe, tmp_path, name):
    make, split, depth = SCENES[name]
    tris = np.ascontiguousarray(make(), np.float32)
    rays = _rays(tris, 4000, seed=len(name))
    tris.tofile(tmp_path / "tris.bin")
    rays.tofile(tmp_path / "rays.bin")
    r = subprocess.run([probe, str(tmp_path / "tris.bin"), str(tmp_path / "rays.bin"), str(split), str(depth)],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr
    _, n, hits, groups, chains = r.stdout.split()
    print(f"[case] {name}: {n} rays, {hits} hits, {groups} groups, {chains} hits in leaves that do not nest")
    assert int(hits) > len(rays) // 50
    if name == "tiny":
        assert int(chains) > 0
