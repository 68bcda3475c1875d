"""Instance casts at the edges of their kernel: ray counts around waves, windows and the persistent
grid, identical instances (equal hits, equal boxes), meshes and top trees deeper than the stack's LDS
part, tMax values at a box's entry, and rays and object-space rays that walk binary nodes. Everything
equals the oracle exactly: the kernel performs its operations in its order."""
import numpy as np
import pytest

from oracle import oracle as O
from phantasyenginetestbed_amd import phx
from test_gpu_instances import aimed_rays, check, ctx, meshes, placed  # noqa: F401
from test_gpu_parity import caterpillar

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 63, 64, 65, 257, 4096, 100003])
@pytest.mark.parametrize("count", [1, 2, 120])
def test_ray_counts(ctx, meshes, count, n):
    specs = placed(meshes, count, 31 + count)
    check(ctx, specs, aimed_rays(specs, np.random.default_rng(n), n))


@pytest.mark.parametrize("copies", [2, 3, 9])
def test_identical_instances(ctx, meshes, copies):
    """The same mesh in the same place several times: every hit ties, the lowest index wins."""
    one = placed(meshes, 1, 5)[0]
    specs = [one] * copies + placed(meshes, 4, 6)
    _, ids, _ = check(ctx, specs, aimed_rays(specs, np.random.default_rng(copies), 9001))
    assert (ids == 0).sum() > 100 and not np.isin(ids, range(1, copies)).any()


def test_limits_at_box_entries(ctx, meshes):
    """tMax equal to, just below and just above the closest hit: the last box that may still be
    entered."""
    specs = placed(meshes, 60, 8)
    rays = aimed_rays(specs, np.random.default_rng(2), 6000)
    rays["tmax"] = np.float32(phx.FLT_MAX)
    hits, _ = O.cast_instances([(b.nodes, b.tris, m) for b, _, m in specs], rays)
    t = hits["t"][hits["tri"] != phx.MISS]
    rays = rays[hits["tri"] != phx.MISS]
    for lim in (t, np.nextafter(t, np.float32(0)), np.nextafter(t, np.float32(np.inf))):
        r = rays.copy()
        r["tmax"] = lim
        check(ctx, specs, r)
    for lim in (0.0, -0.0, -1.0, np.inf, np.nan):
        r = rays[:500].copy()
        r["tmax"] = np.float32(lim)
        check(ctx, specs, r)


def test_axis_aligned_rays(ctx, meshes):
    """Zero direction components in world space, and in object space under unrotated instances."""
    specs = placed(meshes, 20, 9)
    for i in range(0, 20, 2):
        m = np.zeros((3, 4), np.float32)
        m[:, :3] = np.diag([1.0, 2.0, 0.5])
        m[:, 3] = specs[i][2][:, 3]
        specs[i] = (*specs[i][:2], m)
    rays = aimed_rays(specs, np.random.default_rng(4), 5000)
    rays["d"][::2, 1] = 0.0
    rays["d"][::3, 2] = -0.0
    with np.errstate(all="ignore"):
        check(ctx, specs, rays)


@pytest.mark.parametrize("count", [1, 40])
def test_deep_meshes(ctx, count):
    """A mesh 60 levels deep: pending entries beyond the LDS rows, above the top tree's."""
    nodes, tris = caterpillar()
    s = ctx.upload_scene(nodes, tris)

    class Mesh:
        pass
    b = Mesh()
    b.nodes, b.tris = nodes, tris
    rng = np.random.default_rng(12)
    specs = []
    for _ in range(count):
        m = np.zeros((3, 4), np.float32)
        m[:, :3] = np.linalg.qr(rng.normal(size=(3, 3)))[0]
        m[:, 3] = rng.uniform(-2, 2, 3)
        specs.append((b, s, m))
    try:
        check(ctx, specs, aimed_rays(specs, rng, 3000))
    finally:
        s.release()
