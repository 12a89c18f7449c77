"""The 256-channel LayerNorm tiles: each tile width (8, 16 and 32 pixels, by
the plane's size), planes that end inside a tile, and one off the 128-bit path,
to the bit of the one-pass fp32 LayerNorm of the CPU path."""

import numpy as np
import pytest

from test_gpu_pointwise import oracle_plan, run_plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,w,kernel", [
    (1, 4, "mx_chan_ln_c256_p8"),
    (28, 45, "mx_chan_ln_c256_p8"),       # 1260 pixels: half a tile at the end
    (92, 91, "mx_chan_ln_c256_p16"),      # 8372 pixels, a quarter of a tile
    (130, 130, "mx_chan_ln_c256"),        # 16900 pixels, an eighth
    (13, 21, "mx_chan_ln_any"),           # rows not a multiple of 4 pixels
])
def test_layernorm_of_256_channels(gpu_ok, h, w, kernel):
    from maxim_amd import plan as P
    rng = np.random.default_rng(h + w)
    x = (rng.standard_normal((256, h, w)) + 2).astype(np.float32)
    s = rng.standard_normal(256).astype(np.float32)
    b = rng.standard_normal(256).astype(np.float32)
    op = P.make_op(P.CHAN_LN, dst=1, src=0, scale=0, bias=1, c=256, hw=h * w)
    cp = P.CustomPlan([(256, h, w), (256, h, w)], [op], [s, b], input=0, output=1)
    got, steps = run_plan(cp, {0: x}, 1)
    print(h, w, steps, flush=True)
    assert steps[0][2] == kernel
    assert np.array_equal(got.view(np.uint32), oracle_plan(cp, {0: x}, 1).reshape(got.shape).view(np.uint32))
