"""Casts and requests on host memory: arrays around the size up to which the kernels read them in
place, and requests whose rays and outputs are pinned, pageable, misaligned or odd in length, more of
them than one copy launch takes. Compared exactly with the oracle; bytes beside an output stay."""
import time

import numpy as np
import pytest

from oracle import oracle as O
from phantasyenginetestbed_amd import phx

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = phx.Context(0)
    yield c
    c.destroy()


@pytest.fixture(scope="module")
def scene(ctx):
    t, d = phx.random_triangles(4000, 21, 0.02, 0.2)
    b = phx.BVH(t, d)
    s = ctx.upload_scene(b.nodes, b.tris, b.datas)
    yield b, s
    s.release()


def some_rays(n, seed):
    rng = np.random.default_rng(seed)
    rays = np.zeros(n, phx.RAY)
    rays["o"] = rng.uniform(-0.2, 1.2, (n, 3)).astype(np.float32)
    d = rng.normal(size=(n, 3))
    rays["d"] = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    rays["tmin"], rays["tmax"] = np.float32(1e-4), np.float32(phx.FLT_MAX)
    return rays


@pytest.mark.parametrize("kernel", [0, phx.KERNEL_ONE_RAY_PER_LANE, phx.KERNEL_PACKET])
@pytest.mark.parametrize("n", [1, 2, 1000, 8191, 8192, 8193, 20000])
def test_host_casts(ctx, scene, n, kernel):
    b, s = scene
    rays = some_rays(n, n)
    hits, lit = O.cast_closest(b.nodes, b.tris, rays), O.cast_anyhit(b.nodes, b.tris, rays)
    for _ in range(2):
        assert ctx.cast_closest(s, rays, kernel).tobytes() == hits.tobytes()
        assert (ctx.cast_anyhit(s, rays, kernel) == lit).all()
    assert ctx.cast_closest(s, rays[:0], kernel).size == 0


@pytest.mark.parametrize("slots", [1, 3])
@pytest.mark.parametrize("memory", ["pinned", "pageable", "shifted", "mixed"])
def test_requests(ctx, scene, memory, slots):
    """150 requests; "shifted": rays 4 and outputs 1 byte (flags) or 4 bytes (hits) past an aligned
    address of pinned memory."""
    b, s = scene
    rng = np.random.default_rng(slots)
    server = phx.Server(ctx, 1 << 30, slots=slots)
    server.add_scene(s)
    jobs, keep = [], []
    try:
        for i in range(150):
            how = memory if memory != "mixed" else ["pinned", "pageable", "shifted"][i % 3]
            n = int(rng.integers(1, 4000)) if i % 5 else i % 17 + 1
            rays, anyhit = some_rays(n, i), i % 2 == 1
            shift, size = (1 if anyhit else 4) if how == "shifted" else 0, n if anyhit else 16 * n
            nbytes = 32 * n + 8, size + 32
            if how == "pageable":
                rb, ob = np.zeros(nbytes[0], np.uint8), np.zeros(nbytes[1], np.uint8)
            else:
                bufs = [phx.HostBuffer(np.uint8, k) for k in nbytes]
                keep += bufs
                rb, ob = bufs[0].array, bufs[1].array
            at = 4 if how == "shifted" else 0
            rb[at:at + 32 * n] = rays.view(np.uint8).ravel()
            ob[:] = 0xA5
            kind = phx.BATCH_ANYHIT if anyhit else phx.BATCH_CLOSEST
            req = phx.Server.request(s, rb.ctypes.data + at, ob.ctypes.data + shift, n, kind)
            jobs.append((rb, ob, shift, size, rays, anyhit, server.submit(req)))
        for rb, ob, shift, size, rays, anyhit, ticket in jobs:
            limit = time.monotonic() + 30
            while not server.poll(ticket)[0]:
                assert time.monotonic() < limit
                time.sleep(0.0005)
            ref = (O.cast_anyhit if anyhit else O.cast_closest)(b.nodes, b.tris, rays)
            assert ob[shift:shift + size].tobytes() == ref.tobytes(), (len(rays), anyhit)
            assert (ob[:shift] == 0xA5).all() and (ob[shift + size:] == 0xA5).all()
    finally:
        server.destroy()
        jobs.clear()
        rb = ob = None
        for k in keep:
            k.free()
