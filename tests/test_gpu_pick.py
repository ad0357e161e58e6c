"""GPU: picking (st_pick) against the oracle's restatement of
manipulateSelection's pick branch (viewport/manipulation.h:55-124), which
tests/test_pick_oracle.py pins to the reference's own code: object type
and id, hit point and view-space distance bit for bit, on the example
scenes, a mesh scene and points on light glow spheres."""
from __future__ import annotations

import numpy as np
import pytest

import checkers as ck
import scenes
import slimtracin_amd as st
from slimtracin_amd.scene import (IS_ROTATED, MODE_NORMALS, PRIM_LIGHT, blob_mesh_info, blob_prims,
                                  blob_with_prebuilt_meshes, blob_with_prims, make_view)

pytestmark = pytest.mark.gpu

CASES = ["ex01_lights", "ex02_geometry", "ex04_glass_mirror", "ex06_area_lights", "ex07_monkey", "ex09_textures"]


def _grid(w, h, step):
    ys, xs = np.mgrid[0:h + 1:step, 0:w + 1:step]
    return np.stack([xs.ravel(), ys.ravel()], axis=1).astype(np.uint32)


@pytest.mark.parametrize("name", CASES)
def test_pick_matches_oracle(name):
    st.init(0)
    s, cam = getattr(scenes, name)()
    blob = s.to_blob()
    view = make_view(width=200, height=150, **cam)
    xy = _grid(200, 150, 2)
    ds = st.DeviceScene(blob)
    try:
        got = st.pick(ds, view, xy)
    finally:
        ds.close()
    want = ck.oracle_pick(blob, view, xy)
    same = got.view(np.uint8).reshape(len(xy), -1) == want.view(np.uint8).reshape(len(xy), -1)
    rows = np.nonzero(~same.all(axis=1))[0]
    print(name, "points", len(xy), "hits", int((got["object_type"] > 0).sum()), "mismatches", len(rows), flush=True)
    assert len(rows) == 0, (name, xy[rows[:4]], got[rows[:2]], want[rows[:2]])


def test_pick_lights_and_mesh_scene():
    st.init(0)
    s, cam = scenes.ex01_lights()
    blob = s.to_blob()
    view = make_view(width=96, height=72, **cam)
    ds = st.DeviceScene(blob)
    try:
        xy = _grid(96, 72, 1)
        got = st.pick(ds, view, xy)
    finally:
        ds.close()
    want = ck.oracle_pick(blob, view, xy)
    assert got.tobytes() == want.tobytes()
    assert (got["object_type"] == PRIM_LIGHT).any()
    blob = st.gen_pbr(3, 30)
    view = make_view(width=128, height=96, position=(0.0, 6.0, -14.0), pitch=-0.15)
    ds = st.DeviceScene(blob)
    try:
        xy = _grid(128, 96, 2)
        got = st.pick(ds, view, xy)
    finally:
        ds.close()
    want = ck.oracle_pick(blob, view, xy)
    assert got.tobytes() == want.tobytes()


# a whole row and column (with the camera turned a quarter, a column) of rays with an exactly zero direction
# component through an unrotated mesh; the oracle counts thousands of steps for most of them
AXIS_VIEWS = [dict(position=(0.0, 3.0, -10.0), width=33, height=21),
              dict(position=(0.0, 3.0, -10.0), width=65, height=49),
              dict(position=(10.0, 3.0, 0.0), yaw=1.0, width=45, height=27)]


@pytest.mark.parametrize("builder", ["sah", "lbvh"])
@pytest.mark.parametrize("triangles", [500, 4500, 20000])
@pytest.mark.parametrize("k", range(len(AXIS_VIEWS)))
def test_pick_degenerate_rays(k, triangles, builder):
    """Picking has no redo stage: a ray whose traversal is long is traced to its end where it is (meshes below and above
    the size that the redo stage shares out)."""
    blob = st.gen_mesh_scene(5, triangles)
    prims = blob_prims(blob)
    prims[0]["rotation"] = (0.0, 0.0, 0.0, 1.0)
    prims[0]["flags"] &= ~np.uint32(IS_ROTATED)
    blob = want_blob = blob_with_prims(blob, prims)
    if builder == "lbvh":
        T = blob_mesh_info(blob)[0]["triangle_count"]
        want_blob = blob_with_prebuilt_meshes(blob, [ck.oracle_mesh_lbvh(blob, 0, T)])
    view = make_view(**AXIS_VIEWS[k])
    xy = _grid(AXIS_VIEWS[k]["width"], AXIS_VIEWS[k]["height"], 1)
    ds = st.DeviceScene(blob, mesh_lbvh=builder == "lbvh")
    try:
        got = st.pick(ds, view, xy)
    finally:
        ds.close()
    want = ck.oracle_pick(want_blob, view, xy)
    if triangles > 4096:
        steps = ck.oracle_render_steps(want_blob, make_view(mode=MODE_NORMALS, **AXIS_VIEWS[k]))[2]
        assert (steps > 1000).sum() > 10   # traced to the end, more than ten times the limit of the main stages
    assert (want["object_type"] > 0).any()
    assert got.tobytes() == want.tobytes()
