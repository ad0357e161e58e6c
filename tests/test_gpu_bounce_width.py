"""GPU: the bounce stage cuts a short queue into chunks of at least 64, 16 or
4 pixels by what a launch's scenes hold; a frame does not depend on the cut,
so each scene alone equals the same request in a launch of all of them."""
from __future__ import annotations

import numpy as np
import pytest

import slimtracin_amd as st
from slimtracin_amd.scene import MODE_BEAUTY, make_view

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(1, 1), (63, 33), (320, 200)])
def test_chunk_widths_agree(size):
    # 320 and 18,000 triangles; 16 primitives; 4 instances
    blobs = [st.gen_pbr(3, 4), st.gen_pbr(3, 30), st.gen_implicit(3), st.gen_instanced(3, 4, [500, 2000, 5000], 64)]
    scenes = [st.DeviceScene(b, mesh_binned=True) for b in blobs]
    view = make_view(width=size[0], height=size[1], mode=MODE_BEAUTY, depth=5, position=(0.0, 3.0, -9.0), pitch=-0.1)
    try:
        alone = [st.render(s, view) for s in scenes]
        together, _, counts = st.render_batch(scenes, np.concatenate([view] * 4))
        for (pixels, _, c), p, k in zip(alone, together, counts):
            assert pixels.tobytes() == p.tobytes()
            assert (c.primary, c.shadow, c.bounce) == (k.primary, k.shadow, k.bounce)
    finally:
        for s in scenes:
            s.close()
