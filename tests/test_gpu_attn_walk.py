"""GPU: the decode step's exact attention walk (oh_k_attn_walk) at the edges of
its 16-position tiles, its chunks of 7 tiles and its ring of 8 chunks, and at the
last context it takes, against the oracle's ornith_gqa_step
(src/ornith_attn.c:87-149) over the same Q8 KV cache. It adds in the
reference's order: bit-identical."""
import numpy as np
import pytest

import clibs
from test_gpu_attn_parity import C3H, check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,limit", [(64, 3072), (128, 6144), (256, 8192)])
def test_walk_at_tile_and_chunk_edges(hip_ctx, orc, hd, limit):
    cfg = dict(C3H, hd=hd)
    m = hip_ctx.synth(**cfg)
    prompt = clibs.ids(32, "walk.prompt", limit, cfg["vocab"])
    s = m.session(limit)
    for stop in (1, 15, 111, 223, 447, 895, limit - 2):
        s.eval(prompt[s.pos:stop])
        for _ in range(2):                # contexts stop + 1 and stop + 2: an edge's last and first
            s.step(int(prompt[s.pos]))
            o, ref, pos = check(orc, s, cfg, -1)
            assert np.array_equal(o.view(np.uint32), ref.view(np.uint32)), pos + 1
    assert pos + 1 == limit
    s.free()
    m.free()
