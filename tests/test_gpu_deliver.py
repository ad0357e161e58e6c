"""GPU: outputs in page-locked memory (the device writes them itself) equal the same launch's outputs in pageable memory (copied):
grids, hit records and window images of odd sizes, from one pixel up to more
than one block's share, at every 4-byte offset, next to bytes that must stay
as they are."""
from __future__ import annotations

import ctypes as C
import threading

import numpy as np
import pytest

import slimtracin_amd as st
from slimtracin_amd.scene import HIT_DTYPE, MODE_BEAUTY, MODE_DEPTH, MODE_NORMALS, MODE_UVS, PIXEL_DTYPE, make_view
from slimtracin_amd.server import OUTPUT_BGRA8, Server

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (1, 7), (2, 1), (3, 3), (5, 2), (63, 17), (1023, 1), (1025, 3), (333, 41)]


def _views():
    return np.concatenate([make_view(width=w, height=h, mode=MODE_BEAUTY if i % 2 else MODE_NORMALS, depth=2,
                                     position=(0.0, 7.0, -11.0), pitch=-0.2) for i, (w, h) in enumerate(SIZES)])


@pytest.fixture(scope="module")
def scene():
    ds = st.DeviceScene(st.gen_implicit(3))
    yield ds
    ds.close()


def _guarded(sizes, item, offset):
    """Byte slices of one page-locked block at `offset` into a 16-byte grid, guard bytes between them."""
    at, spans = offset, []
    for n in sizes:
        spans.append((at, at + n * item))
        at += n * item + 12
        at += (offset - at) % 16
    block = st.pinned_empty(at + 64, np.uint8)
    block[:] = 0xA5
    return block, spans


def _guards_stand(block, spans):
    outside = np.ones(len(block), bool)
    for a, b in spans:
        outside[a:b] = False
    return bool((block[outside] == 0xA5).all())


@pytest.mark.parametrize("offset", [0, 4, 8, 12])
def test_window_images(scene, offset):
    views = _views()
    want, _ = st.render_batch_bgra8([scene] * len(views), views)
    block, spans = _guarded([w * h for w, h in SIZES], 4, offset)
    outs = [block[a:b].view(np.uint32) for a, b in spans]
    got, counts = st.render_batch_bgra8([scene] * len(views), views, outs=outs)
    for g, w in zip(got, want):
        assert (g == w).all()
    assert _guards_stand(block, spans)
    assert [c.primary for c in counts] == [(w + 1) * (h + 1) for w, h in SIZES]


@pytest.mark.parametrize("offset", [0, 4, 8])
@pytest.mark.parametrize("call", ["batch", "plain", "noalloc"])
def test_grids_and_hits(scene, offset, call):
    views = _views()
    n = len(views)
    grid = [(w + 1) * (h + 1) for w, h in SIZES]
    want_p, want_h, want_c = st.render_batch([scene] * n, views, hits=True)
    pb, ps = _guarded(grid, PIXEL_DTYPE.itemsize, offset)
    hb, hs = _guarded(grid, HIT_DTYPE.itemsize, offset)
    pix = [pb[a:b].view(PIXEL_DTYPE) for a, b in ps]
    hits = [hb[a:b].view(HIT_DTYPE) for a, b in hs]
    counts = (st.RayCounts * n)()
    L = st.lib()
    if call == "batch":
        handles = (C.c_void_p * n)(*[scene.handle] * n)
        rc = L.st_render_batch(handles, views.ctypes.data_as(C.c_void_p), C.c_uint32(n),
                               (C.c_void_p * n)(*[p.ctypes.data for p in pix]),
                               (C.c_void_p * n)(*[h.ctypes.data for h in hits]), counts, C.c_uint32(1))
        assert rc == 0
    else:
        fn = L.st_render if call == "plain" else L.st_render_noalloc
        for i in range(n):
            assert fn(scene.handle, views[i:i + 1].ctypes.data_as(C.c_void_p), C.c_void_p(pix[i].ctypes.data),
                      C.c_void_p(hits[i].ctypes.data), C.byref(counts[i])) == 0
    for i in range(n):
        assert pix[i].tobytes() == want_p[i].tobytes() and hits[i].tobytes() == want_h[i].tobytes()
        assert (counts[i].shadow, counts[i].bounce) == (want_c[i].shadow, want_c[i].bounce)
    assert _guards_stand(pb, ps) and _guards_stand(hb, hs)


@pytest.mark.parametrize("abandon", [0, 48])
@pytest.mark.parametrize("call", ["windows", "grids"])
def test_plain_requests_of_a_mixed_launch(call, abandon):
    """Window images without a bounce stage are delivered while the Beauty requests render, the pixels that the redo
    stage then changes (abandon: a small step limit makes some) once more; grids and hit records are
    written by the stages. Each request alone has none to overlap with."""
    ds = st.DeviceScene(st.gen_pbr(3, 20), mesh_lbvh=True)
    sizes = [(1201, 701), (1, 1), (1600, 900), (640, 363), (1601, 900), (17, 5), (1024, 640)]
    modes = [MODE_BEAUTY, MODE_NORMALS, MODE_NORMALS, MODE_DEPTH, MODE_BEAUTY, MODE_BEAUTY, MODE_UVS]
    if call == "windows":   # enough bytes that the images go out early; grids and hit records always do
        sizes += [(3201, 2003), (3199, 1999), (1601, 1001)]   # (and enough pixels with a bounce stage to do so)
        modes += [MODE_UVS, MODE_NORMALS, MODE_BEAUTY]
    grid = [(w + 1) * (h + 1) for w, h in sizes]
    views = np.concatenate([make_view(width=w, height=h, mode=m, depth=0 if w == 17 else 2,
                                     position=(0.0, 3.0, -9.0), pitch=-0.1) for (w, h), m in zip(sizes, modes)])
    n = len(views)
    try:
        st.debug_redo(abandon, 1 if abandon else 0)
        redone = 0
        if call == "windows":
            want, want_c = [], []
            for i in range(n):
                a, c = st.render_batch_bgra8([ds], views[i:i + 1])
                redone += st.last_redo_count()
                want.append(a[0])
                want_c += c
            block, spans = _guarded([w * h for w, h in sizes], 4, 4)
            outs = [block[a:b].view(np.uint32) for a, b in spans]
            got, counts = st.render_batch_bgra8([ds] * n, views, outs=outs)
            assert all((g == w).all() for g, w in zip(got, want))
            assert _guards_stand(block, spans)
        else:
            want_p, want_h, want_c = [], [], []
            for i in range(n):
                p, h, c = st.render_batch([ds], views[i:i + 1], hits=True)
                redone += st.last_redo_count()
                want_p += p
                want_h += h
                want_c += c
            pb, ps = _guarded(grid, PIXEL_DTYPE.itemsize, 8)
            hb, hs = _guarded(grid, HIT_DTYPE.itemsize, 8)
            pix = [pb[a:b].view(PIXEL_DTYPE) for a, b in ps]
            hits = [hb[a:b].view(HIT_DTYPE) for a, b in hs]
            counts = (st.RayCounts * n)()
            rc = st.lib().st_render_batch((C.c_void_p * n)(*[ds.handle] * n), views.ctypes.data_as(C.c_void_p),
                                          C.c_uint32(n), (C.c_void_p * n)(*[p.ctypes.data for p in pix]),
                                          (C.c_void_p * n)(*[h.ctypes.data for h in hits]), counts, C.c_uint32(1))
            assert rc == 0
            for i in range(n):
                assert pix[i].tobytes() == want_p[i].tobytes() and hits[i].tobytes() == want_h[i].tobytes()
            assert _guards_stand(pb, ps) and _guards_stand(hb, hs)
        assert [(c.primary, c.shadow, c.bounce) for c in counts] == [(c.primary, c.shadow, c.bounce) for c in want_c]
        assert not abandon or redone
    finally:
        st.debug_redo(0, 0)
        ds.close()


def test_mixed_launches_on_two_contexts_while_the_tuning_changes():
    """A server's launches of plain and Beauty requests, split and not, two at a time, while another thread sets the
    claim order: every image equals the one that a launch of its own gives."""
    ds = st.DeviceScene(st.gen_pbr(3, 30), mesh_lbvh=True)
    cam = dict(position=(0.0, 3.0, -9.0), pitch=-0.1)
    kinds = [(2049, 1601, MODE_NORMALS), (1601, 901, MODE_BEAUTY), (2049, 1601, MODE_DEPTH), (1601, 901, MODE_BEAUTY)]
    views = np.concatenate([make_view(width=w, height=h, mode=m, depth=2, **cam) for w, h, m in kinds])
    want = [st.render_batch_bgra8([ds], views[i:i + 1])[0][0] for i in range(len(views))]
    tuned = st.get_tuning()
    srv = Server(output=OUTPUT_BGRA8, max_in_flight=2, max_batch_requests=16)
    done = threading.Event()

    def retune():
        other = st.get_tuning()
        while not done.is_set():
            other.cost_order = 1 - other.cost_order
            st.restore_tuning(other)
            done.wait(0.0003)

    th = threading.Thread(target=retune)
    try:
        sid = srv.add_scene(st.gen_pbr(3, 30), mesh_lbvh=True)
        th.start()
        tickets = [srv.submit(sid, views[i % 4:i % 4 + 1]) for i in range(64)]
        for i, t in enumerate(tickets):
            image, _, _ = srv.wait(t, timeout_ms=60000)
            srv.release(t)
            assert np.array_equal(image, want[i % 4]), i
    finally:
        done.set()
        if th.ident:
            th.join()
        st.restore_tuning(tuned)
        srv.close()
        ds.close()


@pytest.mark.parametrize("kind", ["page-locked", "pageable"])
@pytest.mark.parametrize("shift", [0, 1, 40001])
def test_outputs_that_share_memory(scene, kind, shift):
    """Of outputs that overlap the last request's stands, as if the requests had been rendered one after another."""
    w, h, cam = 320, 250, dict(position=(0.0, 7.0, -11.0), pitch=-0.2)
    n = (w + 1) * (h + 1)
    views = np.concatenate([make_view(width=w, height=h, mode=m, depth=2, **cam)
                            for m in (MODE_BEAUTY, MODE_DEPTH, MODE_NORMALS)])
    size = n + 2 * shift
    for dtype, pixels, call in ((PIXEL_DTYPE, n, st.render_batch), (np.uint32, w * h, st.render_batch_bgra8)):
        block = st.pinned_empty(size, dtype) if kind == "page-locked" else np.zeros(size, dtype)
        block.view(np.uint8)[:] = 0
        want = block.copy()
        alone = [call([scene], views[i:i + 1])[0][0] for i in range(3)]
        for i in range(3):
            want[i * shift:i * shift + pixels] = alone[i]
        call([scene] * 3, views, outs=[block[i * shift:i * shift + pixels] for i in range(3)])
        assert block.tobytes() == want.tobytes()
