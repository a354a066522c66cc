"""The device builder's box pyramid joins eight entries at a time, two levels
a pass: its trees at counts around powers of eight and of a wave, byte for
byte against the oracle's."""
import numpy as np
import pytest

import oracle as O
from test_gpu_build import node_bytes, soup_like

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [7, 8, 9, 63, 64, 65, 511, 512, 513, 4095, 4097, 32769, 262145])
@pytest.mark.parametrize("degenerate", [False, True])
def test_tree_bytes(rt, gpu_ctx, n, degenerate):
    t = soup_like(n, n % 97, degenerate=degenerate)
    print(f"case: {n} triangles, degenerate {degenerate}", flush=True)
    want, _, _ = O.lbvh(t)
    assert np.array_equal(node_bytes(gpu_ctx.build_bvh(t)), node_bytes(want))
