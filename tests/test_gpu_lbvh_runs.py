"""GPU: the device LBVH's boxes and nodes where a build's runs of 1024 sorted
leaves end (st_mesh_lbvh.hip merges a run's nodes in LDS and the nodes that
reach over its ends in device memory): sizes around one and two runs, with
all keys different, many equal, and all equal (a run then holds one deep
subtree of keys told apart by their position). Trees equal the oracle's bit
for bit."""
from __future__ import annotations

import numpy as np
import pytest

import checkers as ck
import slimtracin_amd as st
from slimtracin_amd.scene import PRIM_SPHERE, Material, Primitive, Scene, blob_prims, blob_with_prims

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["different", "many equal", "all equal"])
@pytest.mark.parametrize("n", [2, 1023, 1024, 1025, 2047, 2048, 2049, 5000])
def test_lbvh_over_run_ends(n, kind):
    rng = np.random.default_rng(n)
    s = Scene()
    s.materials = [Material()]
    s.primitives = [Primitive(PRIM_SPHERE, position=tuple(rng.uniform(-1, 1, 3)), scale=(0.1, 0.1, 0.1))
                    for _ in range(n)]
    blob = s.to_blob()
    prims = blob_prims(blob)
    span = {"different": 1.0, "many equal": 8.0, "all equal": 0.0}[kind]
    pos = rng.uniform(-1, 1, (n, 3)) if kind == "different" else np.floor(rng.uniform(0, span, (n, 3)))
    prims["position"] = pos.astype(np.float32)
    prims["scale"] = rng.uniform(0.01, 0.2, (n, 1)).astype(np.float32)
    ds = st.DeviceScene(blob)
    try:
        ds.set_prims(prims)
        ds.rebuild(st.ST_REBUILD_LBVH)
        nodes, leaf, h = ds.bvh()
    finally:
        ds.close()
    want_nodes, want_leaf, want_h = ck.oracle_lbvh_build(ck.oracle_prim_boxes(blob_with_prims(blob, prims), n))
    assert h == want_h and (leaf == want_leaf).all()
    assert nodes.tobytes() == want_nodes.tobytes()
