"""GPU: large copies of pageable memory through the ring of page-locked slots
(st_copy.h). Downloads just below, at and above the size where they start, of
whole and broken slots, and once and twice round the ring, equal the same
frames in page-locked memory; a device-built mesh whose indices leave its
arrays is refused wherever the index stands, in small and in large uploads,
and the library goes on."""
from __future__ import annotations

import struct

import numpy as np
import pytest
import torch

import slimtracin_amd as st
from slimtracin_amd.scene import MODE_DEPTH, PIXEL_DTYPE, blob_mesh_info, make_view

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene():
    ds = st.DeviceScene(st.gen_implicit(3))
    yield ds
    ds.close()


# 24-byte pixels: 4 MiB is 174,762.67 of them, a slot 87,381.33, the ring 699,050.67
@pytest.mark.parametrize("w,h", [(417, 417), (418, 417), (599, 291), (1023, 682), (1199, 1165), (1439, 1079)])
def test_downloads(scene, w, h):
    view = make_view(width=w, height=h, mode=MODE_DEPTH, position=(0.0, 7.0, -11.0), pitch=-0.2)
    n = (w + 1) * (h + 1)
    want = st.pinned_empty(n, PIXEL_DTYPE)
    st.render(scene, view, hits=False, out=want)
    for _ in range(2):
        got, hits, _ = st.render(scene, view)
        assert got.tobytes() == want.tobytes()
        assert np.array_equal(hits["prim_id"] >= 0, np.isfinite(want["depth"]))


@pytest.mark.parametrize("tris", [500, 200_000, 600_000])
@pytest.mark.parametrize("which", ["position", "normal"])
@pytest.mark.parametrize("place", ["first", "middle", "last"])
def test_indices_out_of_range_are_refused(tris, which, place):
    blob = bytearray(st.gen_mesh_scene(9, tris))
    m = blob_mesh_info(bytes(blob))[0]
    T, V, N = m["triangle_count"], m["vertex_count"], m["normals_count"]
    at = m["offset"] + 56 + 12 * V
    limit = V
    if which == "normal":
        assert N
        at += 12 * T + 12 * N
        limit = N
    at += 4 * {"first": 0, "middle": 3 * T // 2, "last": 3 * T - 1}[place]
    struct.pack_into("<I", blob, at, limit)
    with pytest.raises(st.SlimTracinError, match="index out of range"):
        st.DeviceScene(bytes(blob), mesh_lbvh=True)
    struct.pack_into("<I", blob, at, limit - 1)
    st.DeviceScene(bytes(blob), mesh_lbvh=True).close()


@pytest.mark.parametrize("whose", ["another library's", "unaligned"])
@pytest.mark.parametrize("w,h", [(599, 291), (1439, 1079)])
def test_downloads_into_page_locked_memory_that_the_device_does_not_write(scene, whose, w, h):
    """Copied directly, next to hit records in pageable memory that take the ring."""
    view = make_view(width=w, height=h, mode=MODE_DEPTH, position=(0.0, 7.0, -11.0), pitch=-0.2)
    n = (w + 1) * (h + 1)
    want, want_hits, _ = st.render(scene, view)
    if whose == "unaligned":
        block = st.pinned_empty(24 * n + 4, np.uint8)
    else:
        block = torch.zeros(24 * n + 4, dtype=torch.uint8, pin_memory=True).numpy()
    for at in (0, 4) if whose != "unaligned" else (4,):
        block[:] = 0x5A
        out = block[at:at + 24 * n].view(PIXEL_DTYPE)
        _, hits, _ = st.render(scene, view, out=out)
        assert out.tobytes() == want.tobytes() and hits.tobytes() == want_hits.tobytes()
        assert (block[:at] == 0x5A).all() and (block[at + 24 * n:] == 0x5A).all()


def test_many_small_downloads(scene):
    """Pageable window images of odd sizes that share the ring's slots equal the page-locked ones."""
    sizes = [(3 + 7 * i % 400, 150 + 11 * i % 300) for i in range(90)] + [(1, 1), (1201, 1000)]
    views = np.concatenate([make_view(width=w, height=h, mode=MODE_DEPTH, position=(0.0, 7.0, -11.0), pitch=-0.2)
                            for w, h in sizes])
    want, _ = st.render_batch_bgra8([scene] * len(sizes), views, outs=st.pinned_split([w * h for w, h in sizes], np.uint32))
    got, _ = st.render_batch_bgra8([scene] * len(sizes), views)
    for i in range(len(sizes)):
        assert np.array_equal(got[i], want[i]), sizes[i]
