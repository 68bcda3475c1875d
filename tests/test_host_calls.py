"""The library's host code without a GPU: its objects linked with a HIP runtime that logs launches,
copies, waits and allocations, and whose device memory the CPU cannot touch (tests/cpp/fake_hip.cpp).
Kernels do not run, so results are not looked at here."""
import ctypes as C
import multiprocessing
import subprocess
import threading
from pathlib import Path

import numpy as np
import pytest

from phantasyenginetestbed_amd import build as pkg_build
from phantasyenginetestbed_amd import phx

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    sources = [p for p in pkg_build.CSRC.iterdir() if p.suffix in (".cpp", ".hip")]
    objects = [pkg_build.BUILD / (p.name + ".o") for p in sources]
    if not all(o.exists() and o.stat().st_mtime >= p.stat().st_mtime
               for o, p in zip(objects, sources)):
        pkg_build.build()
    so = tmp_path_factory.mktemp("host") / "libphx_host.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
                    f"-I{pkg_build.ROCM}/include", str(ROOT / "tests" / "cpp" / "fake_hip.cpp"),
                    *map(str, objects), "-Wl,-Bsymbolic", "-lpthread", "-o", str(so)], check=True)
    return so


def _child(so, test, args, pipe):
    phx.LIB_PATH = Path(so)
    try:
        pipe.send((None, test(phx.lib(), *args)))
    except BaseException as e:  # reported by the parent
        pipe.send((f"{type(e).__name__}: {e}", None))


def run(so, test, *args):
    """test(lib, *args) in a process of its own, with the library at `so`; a crash fails the test."""
    spawn = multiprocessing.get_context("spawn")
    mine, theirs = spawn.Pipe()
    p = spawn.Process(target=_child, args=(str(so), test, args, theirs))
    p.daemon = True
    p.start()
    theirs.close()
    try:
        assert mine.poll(120), "no answer"
        error, result = mine.recv()
    except EOFError:
        p.join()
        pytest.fail(f"the process ended with {p.exitcode}")
    p.join()
    assert error is None, error
    return result


def log(lib) -> list:
    lib.fake_log.restype = C.c_size_t
    out = C.create_string_buffer(1 << 22)
    n = lib.fake_log(out, C.c_size_t(len(out)))
    assert n <= len(out)
    return out.raw[:n].decode().splitlines()


def upload(ctx, n=50, seed=1):
    t, d = phx.random_triangles(n, seed, 0.1, 0.5)
    b = phx.BVH(t, d)
    return ctx.upload_scene(b.nodes, b.tris, b.datas)


def some_rays(n):
    rays = np.zeros(n, phx.RAY)
    rays["d"], rays["tmax"] = 1, 1
    return rays


def traversal_stats(lib, n, mode):
    ctx = phx.Context(0)
    s = upload(ctx)
    ctx.cast_closest(s, some_rays(5))
    log(lib)
    ctx.traversal_stats(s, some_rays(n), mode)
    return log(lib)


@pytest.mark.parametrize("mode", [0, phx.STATS_ANYHIT])
@pytest.mark.parametrize("n", [1, 8192, 8193, 20000])
def test_traversal_stats_of_host_rays_keeps_its_results_on_the_device(library, n, mode):
    """Its hits are device memory: nothing is copied there, by a store or by a call."""
    copies = [x for x in run(library, traversal_stats, n, mode) if x.startswith("copy")]
    assert copies == ([] if n <= 8192 else [f"copy {32 * n} kind=1 {copies[0].split()[-1]}"])


def serve(lib, rays, n, out):
    ctx = phx.Context(0)
    s = upload(ctx)
    server = phx.Server(ctx, 1 << 28)
    server.add_scene(s)
    log(lib)
    try:
        server.wait(server.submit(phx.Server.request(s, rays, out, n, phx.BATCH_CLOSEST)))
        return log(lib)
    finally:
        server.destroy()


def serve_pinned(lib, pins, at, n):
    """A request whose n rays start `at` bytes into memory of which the ranges `pins` are pinned."""
    mem = np.zeros(1 << 20, np.uint8)
    first = mem.ctypes.data + -mem.ctypes.data % 4096
    for lo, hi in pins:
        lib.fake_pin(C.c_void_p(first + lo), C.c_size_t(hi - lo))
    out = np.zeros(n, phx.HIT)
    return serve(lib, first + at, n, out.ctypes.data)


K = 1024


@pytest.mark.parametrize("pins, at, n, in_place", [
    ([(0, 64 * K)], 0, 2048, True),
    ([(0, 64 * K)], 32 * K, 1024, True),
    ([(0, 64 * K)], 32 * K, 1025, False),                     # one ray past the end
    ([(0, 64 * K), (128 * K, 192 * K)], 0, 6144, False),      # pageable memory between two allocations
    ([(0, 64 * K), (64 * K, 128 * K)], 0, 4096, False),       # two allocations side by side
    ([(64 * K, 128 * K)], 64 * K - 32, 2, False),
    ([(0, 64 * K)], 8, 16, False),                            # misaligned
    ([], 0, 64, False)])
def test_only_rays_inside_one_pinned_allocation_are_read_in_place(library, pins, at, n, in_place):
    copies = [x for x in run(library, serve_pinned, pins, at, n) if x.startswith(f"copy {32 * n} kind=1")]
    assert len(copies) == (0 if in_place else 1)


def served_backlog(lib, where):
    """One launch per request: 4 million rays each (2 million: a mixed launch's two requests)."""
    ctx = phx.Context(0)
    s = upload(ctx)
    server = phx.Server(ctx, 1 << 31, slots=4)
    server.add_scene(s)
    n = 4 << 20
    rays, out = phx.HostBuffer(np.uint8, 32 * n), phx.HostBuffer(np.uint8, 16 * n)
    try:
        server.pause()
        tickets = []
        for w in where:
            for part, flags in {"host": [(n, 0)], "device": [(n, phx.MEM_DEVICE)], "empty": [(0, 0), (n, phx.MEM_DEVICE)],
                                "mixed": [(n // 4, 0), (3 * n // 4, phx.MEM_DEVICE)]}[w]:
                tickets.append(server.submit(phx.Server.request(
                    s, rays.array.ctypes.data, out.array.ctypes.data, part, phx.BATCH_ANYHIT, flags)))
        log(lib)
        server.pause(False)
        for t in tickets:
            server.wait(t)
        return log(lib)
    finally:
        server.destroy()


@pytest.mark.parametrize("where, waits", [
    (["host", "host", "host"], [None, 0, 1]),
    (["host", "device", "device"], [None, None, None]),
    (["host", "device", "host"], [None, None, 0]),
    (["device", "host", "host"], [None, None, 1]),
    (["host", "mixed", "empty"], [None, 0, None])])
def test_launches_that_bring_no_rays_wait_for_nobodys(library, where, waits):
    """waits: per launch, the earlier launch whose rays' arrival it waits for."""
    lines = run(library, served_backlog, where)
    launches = [{}]  # per launch, what comes before its traversal: (wait's event, event recorded)
    for x in lines:
        words = dict(w.split("=") for w in x.split() if "=" in w)
        if x.startswith("wait"):
            launches[-1]["waits"] = words["event"]
        elif x.startswith("record") and "traced" not in launches[-1]:
            launches[-1]["loaded"] = words["event"]
        elif "k_trace_batches" in x:
            launches[-1]["traced"] = True
        elif x.startswith("record"):
            launches.append({})
    launches.pop()
    assert len(launches) == len(where)
    loaded = [k.get("loaded") for k in launches]
    assert [k.get("waits") for k in launches] == [None if w is None else loaded[w] for w in waits]


def test_copies_leave_the_link_to_others(library):
    """The reads of a copy kernel that are in flight hold up every other read over the link."""
    lines = run(library, served_backlog, ["host", "device"])
    grids = [int(w[5:]) for x in lines if "k_copy_ranges" in x for w in x.split() if w.startswith("grid=")]
    assert grids == [32, 16, 2]  # rays in, flags out; the device-resident launch's table


def launches(lines, kernel):
    """(grid, block, window, refill) of every launch of `kernel`, in order."""
    out = []
    for x in lines:
        if x.startswith("kernel") and kernel in x:
            w = dict(w.split("=") for w in x.split() if "=" in w)
            out.append(tuple(int(w[k]) for k in ("grid", "block", "window", "refill")))
    return out


def fused(lib, n, refill, fetch, how):
    ctx = phx.Context(0)
    s = upload(ctx)
    rays, out = ctx.alloc(32 * n), ctx.alloc(16 * n)
    ctx.set_launch_params(refill_min=refill, rays_per_fetch=fetch)
    if how == "server":
        server = phx.Server(ctx, 1 << 28)
        server.add_scene(s)
        log(lib)
        try:
            server.wait(server.submit(phx.Server.request(s, rays.ptr, out.ptr, n, phx.BATCH_CLOSEST,
                                                         phx.MEM_DEVICE)))
        finally:
            server.destroy()
        return log(lib)
    if how == "set":  # by hand, after the context's
        ctx.set_launch_params(refill_min=8, rays_per_fetch=64)
    plan = phx.Plan(ctx, [(s, rays.ptr, out.ptr, n, phx.BATCH_CLOSEST)])
    if how == "set":
        plan.set_launch_params(512, block_threads=512, refill_min=refill, rays_per_fetch=fetch)
    log(lib)
    plan.launch()
    return log(lib)


@pytest.mark.parametrize("how", ["context", "set", "server"])
@pytest.mark.parametrize("refill, fetch", [(1, 8), (8, 64), (24, 16), (64, 256)])
def test_fused_launches_take_refill_threshold_and_rays_per_fetch(library, how, refill, fetch):
    """From the plan, or the context that it or the server was made with (the server's rays per fetch:
    the default)."""
    (_, _, window, took), = launches(run(library, fused, 200000, refill, fetch, how), "k_trace_batches")
    assert took == refill and window == (64 if how == "server" else min(fetch, 64))


def tuned(lib, n, plan):
    ctx = phx.Context(0)
    s = upload(ctx)
    rays, out = ctx.alloc(32 * n), ctx.alloc(16 * n)
    p = phx.Plan(ctx, [(s, rays.ptr, out.ptr, n, phx.BATCH_CLOSEST)]) if plan else None
    log(lib)
    p.autotune() if plan else ctx.autotune(s, rays.ptr, n)
    return log(lib)


@pytest.mark.parametrize("plan", [False, True], ids=["cast", "plan"])
@pytest.mark.parametrize("n", [100, 3000, 60000, 4000000])
def test_autotuners_time_no_launch_twice(library, plan, n):
    """Both stages time each of their launch shapes once a round."""
    lines = run(library, tuned, n, plan)
    shapes = launches(lines, "k_trace_batches" if plan else "k_quad")
    reps = (3, 5) if plan else (13, 15)
    # A warm-up and reps rounds of the first stage, then of the second, which has its winner again.
    k = next(i for i in range(1, len(shapes)) if shapes[i] == shapes[0])
    assert len(set(shapes[:k])) == k
    rest = shapes[k * (reps[0] + 1):]
    assert shapes[:k * (reps[0] + 1)] == shapes[:k] * (reps[0] + 1)
    m = len(rest) // (reps[1] + 1)
    assert rest == rest[:m] * (reps[1] + 1) and len(set(rest[:m])) == m
    if n == 4000000:
        assert k == 6 and m == (3 if plan else 1)


def shapes(lib, scenes, track, tries):
    """For each (block, topNodes, helpers, depth): whether the context and a plan over `scenes` take it."""
    ctx = phx.Context(0)
    up = [upload(ctx, n, i + 1) for i, n in enumerate(scenes)]
    mem = ctx.alloc(1 << 16)
    plan = phx.Plan(ctx, [(s, mem.ptr, mem.ptr, 64, phx.BATCH_CLOSEST) for s in up for _ in range(20)], track)

    def takes(f, *a, **k):
        try:
            f(*a, **k)
            return True
        except phx.PhxError as e:
            assert e.status == phx.ERR_INVALID_ARGUMENT
            return False

    return [(takes(ctx.set_launch_params, block_threads=b, top_nodes=top, helper_waves=h, stack_lds_entries=d),
             takes(plan.set_launch_params, 8, block_threads=b, top_nodes=top, helper_waves=h, stack_lds_entries=d))
            for b, top, h, d in tries]


@pytest.mark.parametrize("track", [False, True])
@pytest.mark.parametrize("scenes", [[50], [6000], [50, 60], [6000, 6001]])
def test_shapes_taken_and_refused(library, scenes, track):
    """What a shape stands for has to fit 160 KB of LDS: (depth + 1) x 256 B and 1,440 B a wave, 64 B a
    treelet node, 16 B. In a plan only the nodes count that its one scene has, and its batch table."""
    tries = [(b, top, h, d) for b in (64, 256, 512, 1024) for top in (0, 100, 1000, 1900, 2048)
             for h in (0, 4) for d in (4, 16, 32) if b + 64 * h <= 1024]
    got = run(library, shapes, scenes, track, tries)
    nodes = [len(phx.BVH(*phx.random_triangles(n, i + 1, 0.1, 0.5)).nodes) for i, n in enumerate(scenes)]
    table = 20 * len(scenes) * (16 if track else 4) + 4
    for (b, top, h, d), (by_context, by_plan) in zip(tries, got):
        lds = b // 64 * ((d + 1) * 256 + 1440) + 16
        treelet = min(top, nodes[0]) if len(scenes) == 1 else 0
        assert by_context == (lds + 64 * top <= 163840)
        assert by_plan == (lds + 64 * treelet + table <= 163840), (b, top, h, d)


def resident(lib, block, n):
    ctx = phx.Context(0)
    s = upload(ctx)
    mem = ctx.alloc(32 * n)
    ctx.set_launch_params(block_threads=block, top_nodes=0, helper_waves=0)
    top = ctx.launch_params()["residentGridBlocks"]
    out = []
    for grid in (top // 2, top, top + 9):
        ctx.set_launch_params(grid_closest=grid)
        log(lib)
        ctx.cast_closest_device(s, mem.ptr, n, mem.ptr)
        out += launches(log(lib), "k_quad")
    return out


@pytest.mark.parametrize("block", [64, 256, 512, 1024])
def test_resident_grid_is_where_more_blocks_change_nothing(library, block):
    half, whole, more = run(library, resident, block, 4 << 20)
    assert half[0] < whole[0] and whole == more


def frame_memory(lib, w, h, lights, instances, graph):
    """Device bytes allocated by a frame, with `instances` by those after one without too."""
    ctx = phx.Context(0)
    t, d = phx.random_triangles(50, 1, 0.1, 0.5)
    b = phx.BVH(t, d)
    s = ctx.upload_scene(b.nodes, b.tris, b.datas, phx.materials_random(4, 1), phx.lights_random(lights, 2))
    r = ctx.renderer(w, h)
    cam = phx.camera_look_at((0.5, 0.5, -1.5), (0.5, 0.5, 0), (0, 1, 0), 1.0, w, h)
    image = ctx.alloc(16 * w * h)
    iset = phx.InstanceSet(ctx, [(s, np.eye(3, 4, dtype=np.float32))])
    out = []
    for has in [False, True, False] if instances else [False, False]:
        r.set_instances(iset if has else None)
        log(lib)
        for f in range(2):
            r.render(s, cam, f, 1, phx.FRAME_GRAPH if graph else 0, out_ptr=image.ptr)
        out.append(sum(int(x.split()[1]) for x in log(lib) if x.startswith("malloc")))
    return out


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("w,h,lights", [(64, 32, 8), (33, 17, 3), (1, 9, 2)])
def test_frames_allocate_light_buffers_for_the_records_that_use_them(library, w, h, lights, graph):
    """49 bytes a record and light: the bounce records', and with instances the primary ones'."""
    bounce, primary = (w // 2) * (h // 2) * lights * 49, w * h * lights * 49
    assert run(library, frame_memory, w, h, lights, False, graph) == [bounce, 0]
    assert run(library, frame_memory, w, h, lights, True, graph) == [bounce, primary + 4096, 0]


def cast_windows(lib, n, anyhit, timeline, fetch):
    ctx = phx.Context(0)
    s = upload(ctx)
    ctx.set_launch_params(rays_per_fetch=fetch)
    rays, out = ctx.alloc(32 * n), ctx.alloc(16 * n)
    log(lib)
    if timeline:
        ctx.cast_closest_timeline(s, rays.ptr, n, out.ptr)
    else:
        (ctx.cast_anyhit_device if anyhit else ctx.cast_closest_device)(s, rays.ptr, n, out.ptr)
    return launches(log(lib), "k_quad")


@pytest.mark.parametrize("fetch", [8, 16, 64, 4096])
@pytest.mark.parametrize("n", [1, 2048, 40000, 1 << 20, 16 << 20])
@pytest.mark.parametrize("call", ["closest", "anyhit", "timeline"])
def test_waves_take_no_more_closest_hit_rays_than_they_trace_at_a_time(library, call, n, fetch):
    """A wave traces 16 at a time; rays beside costly ones are costly too, and what is left of a wide window
    is traced by the same wave, one after another."""
    (_, _, window, _), = run(library, cast_windows, n, call == "anyhit", call == "timeline", fetch)
    assert 1 <= window <= min(fetch, 64 if call == "anyhit" else 16)
    if n >= 16 << 20:
        assert window == min(fetch, 64 if call == "anyhit" else 16)


def plan_shapes(lib, sizes):
    ctx = phx.Context(0)
    s = upload(ctx)
    mem = ctx.alloc(32 * max(sizes))
    out = []
    for n in sizes:
        plan = phx.Plan(ctx, [(s, mem.ptr, mem.ptr, n, phx.BATCH_CLOSEST)])
        log(lib)
        plan.launch()
        out += launches(log(lib), "k_trace_batches")
        plan.release()
    return out


def test_small_fused_launches_give_waves_as_many_rays_as_they_trace_four_lanes_each(library):
    sizes = [1, 15, 16, 17, 1000, 65535, 65536, 65537, 4 << 20]
    for n, (grid, block, window, _) in zip(sizes, run(library, plan_shapes, sizes)):
        waves = grid * (block // 64)
        assert window == (16 if n <= 65536 else 64)  # 256 CUs of 16 waves
        assert waves * window >= min(n, 4096 * window) and waves <= 4096


def submit_beside_a_copy(lib):
    """Whether requests are taken while the dispatcher copies, and the launches of all of them."""
    ctx = phx.Context(0)
    s = upload(ctx)
    server = phx.Server(ctx, 1 << 28)
    server.add_scene(s)
    rays, outs = some_rays(256), [np.zeros(256, phx.HIT) for _ in range(9)]
    tickets = []

    def submit(i):
        tickets.append(server.submit(phx.Server.request(s, rays.ctypes.data, outs[i].ctypes.data, 256,
                                                        phx.BATCH_CLOSEST)))

    try:
        lib.fake_hold(1)
        log(lib)
        submit(0)
        while not any(x.startswith("copy") for x in log(lib)):
            pass
        others = threading.Thread(target=lambda: [submit(i) for i in range(1, 9)], daemon=True)
        others.start()
        others.join(5)
        taken = not others.is_alive()
        lib.fake_hold(0)
        others.join()
        for t in tickets:
            server.wait(t)
        return taken, len(launches(log(lib), "k_trace_batches"))
    finally:
        lib.fake_hold(0)
        server.destroy()


def test_requests_are_taken_while_the_dispatcher_copies(library):
    """A copy from pageable memory returns late; what comes meanwhile makes one launch."""
    assert run(library, submit_beside_a_copy) == (True, 2)


def backlog_launches(lib, pinned, count, n):
    ctx = phx.Context(0)
    s = upload(ctx)
    server = phx.Server(ctx, 1 << 30)
    server.add_scene(s)
    make = (lambda k: phx.HostBuffer(np.uint8, k).array) if pinned else (lambda k: np.zeros(k, np.uint8))
    rays, out = make(32 * n), make(n)
    try:
        server.pause()
        tickets = [server.submit(phx.Server.request(s, rays.ctypes.data, out.ctypes.data, n, phx.BATCH_ANYHIT))
                   for _ in range(count)]
        log(lib)
        server.pause(False)
        for t in tickets:
            server.wait(t)
        return launches(log(lib), "k_trace_batches")
    finally:
        server.destroy()


def test_requests_in_pageable_memory_are_not_split(library):
    """Their copy calls return one after another, so nothing overlaps them: launches of up to 4 million
    rays; requests in pinned memory, of a quarter of what waits, a million at least."""
    assert len(run(library, backlog_launches, False, 48, 55000)) == 1
    assert len(run(library, backlog_launches, True, 48, 55000)) == 3


@pytest.mark.parametrize("mode", [0, phx.STATS_ANYHIT])
@pytest.mark.parametrize("n", [1, 1000, 4096, 4097, 20000, 300000])
def test_counting_casts_spread_few_rays_over_the_device(library, n, mode):
    """A wave takes as long as its rays' different steps together: no more rays a wave than 24 waves a CU
    need (256 CUs)."""
    line, = [x for x in run(library, traversal_stats, n, mode) if "simple" in x]
    grid, block = (int(w.split("=")[1]) for w in line.split() if w.startswith(("grid", "block")))
    per_wave = min(64, -(-n // 6144))
    assert -(-n // per_wave) <= grid * (block // 64) < -(-n // per_wave) + 4
