"""The library's host path on the CPU: what it queues, copies and waits for, in which order, over a HIP runtime that
runs no kernels (fake_hip.cpp). Each case runs in a process of its own, with that runtime in place of the real one."""
from __future__ import annotations

import ctypes as C
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CASES = {}


def case(f):
    CASES[f.__name__] = f
    return f


class Fake:
    """The runtime, loaded before the library, and a log of its calls; act(name, args) runs at each of them."""

    def __init__(self, so):
        self.so = C.CDLL(so, mode=C.RTLD_GLOBAL)
        self.so.fake_device_bytes.restype = C.c_size_t
        self.so.fake_host_alloc.restype = C.c_void_p
        self.log, self.act = [], None
        self.hook = C.CFUNCTYPE(None, C.c_char_p, C.POINTER(C.c_void_p))(self._call)
        self.so.fake_hook(self.hook)

    def _call(self, name, args):
        name = name.decode()
        if name.startswith("launch _Z"):   # the kernel's plain name
            digits = "".join(c for c in name[9:12] if c.isdigit())
            name = "launch " + name[9 + len(digits):][:int(digits)]
        self.log.append(name)
        if name == "launch k_mb_emit":   # the height that a device build reports
            C.cast(C.cast(args[5], C.POINTER(C.c_void_p))[0], C.POINTER(C.c_uint32))[0] = 20
        if name == "launch k_deliver":   # the launch's ray counts and fault word
            C.memset(C.cast(args[4], C.POINTER(C.c_void_p))[0], 0, 8 * self.u32(args, 5))
        if self.act:
            self.act(name, args)

    def u32(self, args, i):
        return C.cast(args[i], C.POINTER(C.c_uint32))[0]


def _mixed_batch(st):
    """Requests without a bounce stage with 62 MB of window images and 6 million pixels that have one: a launch that
    is split, the former delivered while the latter render."""
    import numpy as np
    from slimtracin_amd.scene import MODE_BEAUTY, MODE_NORMALS, make_view
    ds = st.DeviceScene(st.gen_pbr(3, 30), mesh_binned=True)
    views = np.concatenate([make_view(width=3839, height=2023, mode=m, depth=3)
                            for m in (MODE_NORMALS, MODE_BEAUTY, MODE_NORMALS)])
    outs = st.pinned_split([3839 * 2023] * 3, np.uint32)
    return [ds] * 3, views, outs


@case
def split_keeps_its_tile_order(fake, st):
    """A launch that is split has its plain requests' tiles first in the claim order; a tuning with an order of its own
    that arrives while the launch is being prepared is for the next one."""
    scenes, views, outs = _mixed_batch(st)
    st.render_batch_bgra8(scenes, views, outs=outs)
    modes = []
    tuned = st.get_tuning()

    def act(name, args):
        if name.startswith("hipOccupancy"):
            tuned.cost_order = 1
            st.restore_tuning(tuned)
        if name == "launch k_prep":
            modes.append(fake.u32(args, 10))

    fake.log.clear()
    fake.act = act
    st.render_batch_bgra8(scenes, views, outs=outs)
    assert fake.log.count("launch k_primary4") == 2, fake.log
    assert modes == [0], modes   # tile order
    del fake.log[:], modes[:]
    for _ in range(2):
        st.render_batch_bgra8(scenes, views, outs=outs)
    assert fake.log.count("launch k_primary4") == 2, fake.log
    assert modes == [0, 1], modes   # slowest first, once this order's times are known


@case
def outputs_that_share_memory_are_copied_in_order(fake, st):
    """Nobody writes such outputs directly, nor with several threads: one copy after another, in the requests' order."""
    import numpy as np
    from slimtracin_amd.scene import MODE_BEAUTY, MODE_DEPTH, PIXEL_DTYPE, make_view
    ds = st.DeviceScene(st.gen_implicit(3))
    w, h = 599, 499
    views = np.concatenate([make_view(width=w, height=h, mode=m, depth=2) for m in (MODE_DEPTH, MODE_BEAUTY, MODE_DEPTH)])
    copies = []
    fake.act = lambda name, args: copies.append((args[0], args[2])) if name == "hipMemcpyAsync" else None
    n = (w + 1) * (h + 1)
    for block in (st.pinned_empty(2 * n, PIXEL_DTYPE), np.empty(2 * n, PIXEL_DTYPE)):
        for outs in ([block[:n], block[n:], block[:n]], [block[:n], block[n // 2:n // 2 + n], block[n:]]):
            del copies[:]
            st.render_batch([ds] * 3, views, outs=outs)
            assert copies == [(o.ctypes.data, 24 * n) for o in outs], copies
    block = st.pinned_empty(2 * w * h + 1, np.uint32)
    for outs in ([block[:w * h]] * 3, [block[1:w * h + 1], block[w * h + 1:], block[:w * h]]):
        del copies[:]
        st.render_batch_bgra8([ds] * 3, views, outs=outs)
        assert copies == [(o.ctypes.data, 4 * w * h) for o in outs], copies
    one = st.pinned_empty(3 * n, PIXEL_DTYPE)
    one = [one[:n], one[n:2 * n], one[2 * n:]]   # neighbours that do not overlap are written by the device
    del copies[:]
    st.render_batch([ds] * 3, views, outs=one)
    assert not copies, copies


@case
def a_failed_call_has_waited_for_its_kernels(fake, st):
    """Whichever call fails after kernels were queued, the stream is waited for before the error is returned."""
    import numpy as np
    from slimtracin_amd.scene import MODE_BEAUTY, PIXEL_DTYPE, make_view
    ds = st.DeviceScene(st.gen_pbr(3, 10))
    view = make_view(width=90, height=70, mode=MODE_BEAUTY, depth=3)
    out = st.pinned_empty(91 * 71, PIXEL_DTYPE)
    xy = np.array([[3, 4], [40, 30]], np.uint32)
    calls = {"render": lambda: st.render(ds, view), "pinned": lambda: st.render(ds, view, hits=False, out=out),
             "noalloc": lambda: st.render_noalloc(ds, view, out=out), "pick": lambda: st.pick(ds, view, xy),
             "graph": lambda: st.render_batch([ds], view, graph=True), "timed": lambda: st.render_timed([ds], view, stages=True),
             "images": lambda: st.render_batch_bgra8([ds], view)}
    failed = 0
    for what, call in calls.items():
        call()
        for name in ("hipGetLastError", "hipMemcpyAsync", "hipEventRecord", "hipGraphLaunch", "hipStreamSynchronize",
                     "hipEventSynchronize"):
            for nth in range(1, 12):
                fake.so.fake_fail(name.encode(), nth)
                del fake.log[:]
                try:
                    call()
                except st.SlimTracinError:
                    failed += 1
                    queued = [i for i, c in enumerate(fake.log) if c.startswith("launch ")]
                    waits = [i for i, c in enumerate(fake.log) if c == "hipStreamSynchronize"]
                    if queued:
                        assert waits and waits[-1] > queued[-1], (what, name, nth, fake.log)
                        assert name != "hipStreamSynchronize" or len(waits) > 1, (what, nth, fake.log)
                else:
                    fake.so.fake_fail(b"", 0)
                    break
    assert failed > 25, failed


def _threads():
    return len(os.listdir("/proc/self/task"))


@case
def copying_threads_start_when_there_is_something_to_copy(fake, st):
    """A large download is queued behind the render; its threads start after the first bytes have arrived, and the call
    takes no processor time of theirs while it waits for the device."""
    import time
    import numpy as np
    from slimtracin_amd.scene import MODE_DEPTH, make_view
    ds = st.DeviceScene(st.gen_implicit(3))
    view = make_view(width=1000, height=700, mode=MODE_DEPTH)
    st.render(ds, view)
    before, seen = _threads(), []

    def act(name, args):
        if name in ("hipEventSynchronize", "hipStreamSynchronize"):
            if not seen:
                t0 = time.process_time()
                time.sleep(0.3)   # the device renders
                seen.append((_threads(), time.process_time() - t0))
            else:
                seen.append((_threads(), 0.0))

    fake.act = act
    st.render(ds, view)
    assert seen[0][0] == before and seen[0][1] < 1.0, (before, seen[0])
    assert max(n for n, _ in seen) > before, seen   # the ring was used


def _each_allocation(fake, st, call, at=None):
    """call() once for each of the library's C++ allocations (from the first `at` on), that one failing: an error or a
    result, and the process goes on. Returns how many there are."""
    for nth in range(1, 400):
        def act(name, args, nth=nth):
            if name == at:
                fake.so.fake_new_fail(nth)
                fake.act = None
        fake.act = act if at else None
        if not at:
            fake.so.fake_new_fail(nth)
        try:
            call()
        except st.SlimTracinError:
            pass
        left = fake.so.fake_new_left()
        fake.so.fake_new_fail(0)
        if left > 0:
            return nth - 1
    raise AssertionError("no end of allocations")


@case
def running_out_of_host_memory_is_an_error(fake, st):
    import numpy as np
    from slimtracin_amd.scene import MODE_BEAUTY, MODE_DEPTH, make_view
    ds = st.DeviceScene(st.gen_implicit(3))
    view = make_view(width=1000, height=700, mode=MODE_DEPTH)
    want = st.render(ds, view)
    assert _each_allocation(fake, st, lambda: st.render(ds, view), at="launch k_deliver") >= 8
    assert _each_allocation(fake, st, lambda: st.render(ds, view)) >= 15
    got = st.render(ds, view)
    assert got[0].tobytes() == want[0].tobytes()
    scenes, views, outs = _mixed_batch(st)
    st.render_batch_bgra8(scenes, views, outs=outs)
    assert _each_allocation(fake, st, lambda: st.render_batch_bgra8(scenes, views, outs=outs)) >= 15
    blob = st.gen_mesh_scene(3, 600000)
    with_meshes = lambda: st.DeviceScene(blob, mesh_lbvh=True).close()   # noqa: E731
    with_meshes()
    bytes_before = fake.so.fake_device_bytes()
    assert _each_allocation(fake, st, with_meshes) >= 8
    assert fake.so.fake_device_bytes() == bytes_before
    assert _each_allocation(fake, st, lambda: st.pinned_empty(100, np.uint8)) >= 1


@case
def a_failed_upload_has_waited_for_its_copies(fake, st):
    """A copy or event of a large upload that fails: the copies before it are waited for before the scene's memory is
    freed or the ring's slots are written again."""
    blob, failed = st.gen_mesh_scene(3, 600000), 0
    for flags in (dict(mesh_binned=True), dict(mesh_lbvh=True)):
        st.DeviceScene(blob, **flags).close()
        for name in ("hipMemcpyAsync", "hipEventRecord", "hipEventSynchronize"):
            for nth in (1, 2, 4, 7):
                fake.so.fake_fail(name.encode(), nth)
                del fake.log[:]
                try:
                    st.DeviceScene(blob, **flags).close()
                    fake.so.fake_fail(b"", 0)   # fewer calls of this kind
                    break
                except st.SlimTracinError:
                    failed += 1
                last = max([i for i, c in enumerate(fake.log) if c == "hipMemcpyAsync"], default=-1)
                after = fake.log[last + 1:]
                assert after.index("hipStreamSynchronize") < after.index("hipFree"), (flags, name, nth, fake.log)
    assert failed > 12, failed


@case
def page_locked_memory_of_others_is_copied_directly(fake, st):
    """Outputs that the device does not write itself but that a copy call can reach at the link's rate: one call each,
    with no threads; pageable ones of the same call still take the ring."""
    import numpy as np
    from slimtracin_amd.scene import HIT_DTYPE, MODE_DEPTH, PIXEL_DTYPE, make_view
    ds = st.DeviceScene(st.gen_implicit(3))
    w, h = 999, 699
    n = (w + 1) * (h + 1)
    view = make_view(width=w, height=h, mode=MODE_DEPTH)
    before, copies, threads = _threads(), [], []

    def act(name, args):
        if name == "hipMemcpyAsync":
            copies.append((args[0], args[2]))
        if name in ("hipEventSynchronize", "hipStreamSynchronize"):
            threads.append(_threads())

    foreign = fake.so.fake_host_alloc(C.c_size_t(24 * n))
    unaligned = st.pinned_empty(24 * n + 4, np.uint8)[4:]
    hits = np.empty(n, HIT_DTYPE)
    st.render(ds, view)
    fake.act = act
    for out in (foreign, unaligned.ctypes.data):
        for hp in (None, hits.ctypes.data):
            del copies[:], threads[:]
            assert st.lib().st_render(ds.handle, C.c_void_p(view.ctypes.data), C.c_void_p(out), C.c_void_p(hp), None) == 0
            assert (out, 24 * n) in copies, copies
            if hp:
                assert len(copies) > 4 and max(threads) > before
            else:
                assert len(copies) == 1 and max(threads) == before


@case
def only_large_copies_take_threads(fake, st):
    """Copies below 4 MiB are plain calls, on the calling thread."""
    from slimtracin_amd.scene import MODE_DEPTH, make_view
    threads = []
    fake.act = lambda name, args: threads.append(_threads())
    before = _threads()
    for triangles, ring in ((60000, False), (100000, True)):
        blob = st.gen_mesh_scene(3, triangles)
        del threads[:]
        st.DeviceScene(blob, mesh_lbvh=True).close()
        assert (max(threads) > before) == ring, (triangles, before, max(threads))
    ds = st.DeviceScene(st.gen_implicit(3))
    for width, ring in ((417, False), (418, True)):
        del threads[:]
        st.render(ds, make_view(width=width, height=417, mode=MODE_DEPTH), hits=False)
        assert (max(threads) > before) == ring, (width, before, max(threads))


@case
def a_mesh_build_keeps_no_device_memory(fake, st):
    """What a device build needs besides the scene is given back before the scene's creation returns."""
    from slimtracin_amd.server import Server
    for triangles in (500, 100000, 600000):
        blob = st.gen_mesh_scene(3, triangles)
        before = fake.so.fake_device_bytes()
        ds = st.DeviceScene(blob, mesh_lbvh=True)
        assert fake.so.fake_device_bytes() - before == ds.info().device_bytes
        ds.close()
        assert fake.so.fake_device_bytes() == before
        srv = Server()
        with_server = fake.so.fake_device_bytes()
        srv.remove_scene(srv.add_scene(blob, mesh_lbvh=True))
        assert fake.so.fake_device_bytes() == with_server
        srv.close()
        assert fake.so.fake_device_bytes() == before
    # a launch buffer that is large enough serves as scratch; one that is not stays as it is
    from slimtracin_amd.scene import MODE_BEAUTY, make_view
    for size, allocations in ((64, 2), (1600, 1)):
        ds = st.DeviceScene(st.gen_implicit(3))
        st.render(ds, make_view(width=size, height=size, mode=MODE_BEAUTY, depth=2))
        ds.close()
        before = fake.so.fake_device_bytes()
        del fake.log[:]
        st.DeviceScene(blob, mesh_lbvh=True).close()
        assert fake.log.count("hipMalloc") == allocations, (size, fake.log)
        assert fake.so.fake_device_bytes() == before


@case
def a_timed_launch_is_timed_from_its_upload_on(fake, st):
    """Launched kernel by kernel or as a graph, the time covers the same work."""
    from slimtracin_amd.scene import MODE_BEAUTY, make_view
    ds = st.DeviceScene(st.gen_pbr(3, 10))
    view = make_view(width=90, height=70, mode=MODE_BEAUTY, depth=3)
    st.render(ds, view)   # the context's arrays are there
    for stages in (False, True):
        for graph in (False, True):
            for _ in range(2):
                del fake.log[:]
                st.render_timed([ds], view, stages=stages, graph=graph)
                work = [i for i, c in enumerate(fake.log) if c == "hipGraphLaunch" or
                        (c.startswith("launch ") and c != "launch k_deliver" and not graph)]
                marks = [i for i, c in enumerate(fake.log) if c == "hipEventRecord"]
                assert marks[0] < work[0] and work[-1] < marks[-1], (stages, graph, fake.log)


@case
def bounce_chunks_by_what_the_scenes_hold(fake, st):
    """The least width of a launch's chunks, by its Beauty requests' scenes as their primitives are now."""
    import numpy as np
    import scenes as examples
    from slimtracin_amd.scene import (MODE_BEAUTY, MODE_DEPTH, PRIM_BOX, PRIM_MESH, blob_prims, blob_with_prims,
                                      make_view)

    def crowd(n, meshes):
        blob = examples.crowd(5, n)[0].to_blob()
        prims = blob_prims(blob)
        prims["type"] = PRIM_BOX
        prims["type"][:meshes] = PRIM_MESH
        return blob_with_prims(blob, prims)

    widths = []
    fake.act = lambda name, args: widths.append(fake.u32(args, 8)) if name == "launch k_bounce" else None
    view = make_view(width=33, height=21, mode=MODE_BEAUTY, depth=3)
    made = {}
    for what, blob, want in [("8", crowd(8, 0), 64), ("15", crowd(15, 3), 64), ("16", crowd(16, 0), 16),
                             ("31", crowd(31, 3), 16), ("32", crowd(32, 0), 4), ("4 meshes", crowd(5, 4), 4),
                             ("320", st.gen_pbr(3, 4), 64), ("18000", st.gen_pbr(3, 30), 16)]:
        ds = made[what] = st.DeviceScene(blob, mesh_binned=True)
        for call in (st.render, st.render_noalloc):
            del widths[:]
            call(ds, view)
            assert widths == [want], (what, widths)
    for names, modes, want in [(("8", "320"), "bb", 64), (("8", "16", "18000"), "bbb", 16), (("8", "32", "320"), "bbb", 4),
                               (("8", "32", "320"), "bdb", 64)]:
        del widths[:]
        st.render_batch([made[n] for n in names], np.concatenate(
            [make_view(width=33, height=21, mode=MODE_BEAUTY if m == "b" else MODE_DEPTH, depth=3) for m in modes]))
        assert widths == [want], (names, widths)
    prims = blob_prims(crowd(5, 3))
    made["4 meshes"].set_prims(np.ascontiguousarray(prims))
    del widths[:]
    st.render(made["4 meshes"], view)
    assert widths == [64], widths


@case
def launches_are_split_when_there_is_enough_to_render_meanwhile(fake, st):
    """By the bytes of the plain requests' images and the pixels, and scenes, of the others."""
    import numpy as np
    from slimtracin_amd.scene import MODE_BEAUTY, MODE_NORMALS, make_view
    heavy, light = (st.DeviceScene(st.gen_pbr(3, k), mesh_binned=True) for k in (30, 4))
    implicit = st.DeviceScene(st.gen_implicit(3))
    block = st.pinned_empty(48 << 20, np.uint32)
    fake.act = None

    def kernels(plain_mb, shaded):
        """Primary kernels of a launch with plain images of so many MiB and Beauty requests (scene, million pixels)."""
        w, h = 4096, round(plain_mb * 2**20 / 4 / 4096)
        views, which, sizes = [make_view(width=w, height=h, mode=MODE_NORMALS)], [implicit], [w * h]
        for ds, mpx in shaded:
            h = round(mpx * 1e6 / 2048)
            views.append(make_view(width=2047, height=h - 1, mode=MODE_BEAUTY, depth=2))
            which.append(ds)
            sizes.append(2047 * (h - 1))
        at = np.concatenate([[0], np.cumsum(sizes)])
        del fake.log[:]
        st.render_batch_bgra8(which[::-1], np.concatenate(views[::-1]), outs=[block[at[i]:at[i + 1]] for i in range(len(sizes))][::-1])
        return fake.log.count("launch k_primary4")

    mb = 2**20 / 1e6
    assert kernels(47.9, [(heavy, 2.0)]) == 1
    assert kernels(48.1, [(heavy, 48.1 * mb / 32 + 0.01)]) == 2
    assert kernels(60.0, [(heavy, 60.0 * mb / 32 - 0.01)]) == 1
    assert kernels(60.0, [(light, 60.0 * mb / 20 - 0.01)]) == 1
    assert kernels(60.0, [(light, 60.0 * mb / 20 + 0.01)]) == 2
    assert kernels(60.0, [(light, 30.0 * mb / 20 + 0.01), (heavy, 30.0 * mb / 32 + 0.01)]) == 2
    assert kernels(48.1, [(implicit, 16.0)]) == 1


@case
def small_spans_share_the_slots_of_the_copy_ring(fake, st):
    """Many small pageable outputs of one launch go slot by slot (2 MiB, an event each), and each arrives whole."""
    import numpy as np
    from slimtracin_amd.scene import MODE_DEPTH, make_view
    ds = st.DeviceScene(st.gen_implicit(3))
    sizes = [(3 + 7 * i % 400, 150 + 11 * i % 300) for i in range(90)] + [(1, 1), (1201, 1000)]
    views = np.concatenate([make_view(width=w, height=h, mode=MODE_DEPTH) for w, h in sizes])
    sent = []

    def act(name, args):   # the device's bytes of each copy: its number
        if name == "hipMemcpyAsync":
            C.memset(args[1], len(sent) % 251 + 1, args[2])
            sent.append(args[2])

    outs = [np.zeros(w * h, np.uint32) for w, h in sizes]
    st.render_batch_bgra8([ds] * len(sizes), views, outs=outs)
    fake.act = act
    del fake.log[:]
    st.render_batch_bgra8([ds] * len(sizes), views, outs=outs)
    total = sum(4 * w * h for w, h in sizes)
    assert sum(sent) == total > 8 << 20
    assert fake.log.count("hipEventRecord") <= total // (2 << 20) + 2, fake.log.count("hipEventRecord")
    at = 0
    for o in outs:
        b, done = o.view(np.uint8), 0
        while done < len(b):
            assert (b[done:done + sent[at]] == at % 251 + 1).all(), at
            done += sent[at]
            at += 1
    assert at == len(sent)


@case
def nothing_is_filled_behind_a_launchs_back(fake, st):
    """hipMemset returns before its fill is done, on a stream that nothing orders against a context's own: a context's
    words and tile arrays are cleared by kernels on its stream, before the launch that uses them."""
    from slimtracin_amd.scene import MODE_BEAUTY, make_view
    from slimtracin_amd.server import Server
    blob = st.gen_implicit(3)
    ds = st.DeviceScene(blob)
    srv = Server(max_in_flight=2)
    sid = srv.add_scene(blob)
    assert fake.log.count("launch k_zero_u32") == 3, fake.log   # the main context and the server's two
    for size in (64, 900, 300, 1200):
        view = make_view(width=size, height=size, mode=MODE_BEAUTY, depth=2)
        del fake.log[:]
        st.render(ds, view)
        grown = fake.log.count("launch k_zero_u32")
        assert grown == (size != 300), fake.log
        if grown:
            assert fake.log.index("launch k_zero_u32") < fake.log.index("launch k_setup")
        t = srv.submit(sid, view)
        srv.wait(t, copy=False)
        srv.release(t)
        assert "hipMemset" not in fake.log, fake.log
    srv.close()


@pytest.fixture(scope="module")
def fake_so(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", os.path.join(HERE, "fake_hip.cpp"), "-o", so],
                   check=True)
    return so


@pytest.mark.parametrize("name", sorted(CASES))
def test_host_path(fake_so, name):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), fake_so, name], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, (r.returncode, r.stdout[-2000:], r.stderr[-4000:])


if __name__ == "__main__":
    sys.path[:0] = [os.path.dirname(HERE), HERE]
    runtime = Fake(sys.argv[1])
    import slimtracin_amd as library
    library.init(0)
    CASES[sys.argv[2]](runtime, library)
    runtime.act = None
