"""The net's kernels over the tiles that their rules choose (k_net.hip: launch_conv, wgrad_shape), against the FP64
oracle with the same BF16 roundings; the bounds are those of test_net: 2e-3 on the image, 2e-2 on a layer's gradient.
"""
from __future__ import annotations

import numpy as np
import pytest

from test_net import _layer_ranges, _params, _problem

pytestmark = pytest.mark.gpu


# the smallest grid (coarsest level one voxel), partial tiles in every direction (widths that are no multiple of 16,
# heights and depths off the tiles of a level), and a grid that fills the chip: the wide tiles at the fine levels, the
# narrow ones at the coarse, several tiles to a gradient partial
@pytest.mark.parametrize("shape", [(8, 8, 8), (8, 24, 40), (24, 16, 136), (40, 72, 24), (32, 128, 128)])
def test_net_matches_oracle_on_every_tile(oracle, shape):
    from pct_reconstruction_amd.learned import WarmStartNet
    fbp, hull, target = _problem(shape, 21)
    p = _params(oracle, 22)
    ref_loss, ref_g, ref_x0 = oracle.net_loss_grad(shape, p, fbp, hull, target, bf16=True)
    with WarmStartNet(shape[2], shape[1], shape[0], seed=0) as net:
        net.set_params(p)
        x0 = net.predict(fbp, hull)
        loss, g = net.loss_grad(fbp, hull, target)
    print(f"{shape}: loss gpu {loss:.6e} oracle {ref_loss:.6e}", flush=True)
    assert abs(loss - ref_loss) <= 2e-3 * ref_loss
    assert np.linalg.norm(x0 - ref_x0) <= 2e-3 * np.linalg.norm(ref_x0)
    weights = _layer_ranges()
    ends = [a for a, _ in weights[1:]] + [p.size]
    for k, ((a, b), e) in enumerate(zip(weights, ends)):
        for kind, lo, hi in (("weights", a, b), ("biases", b, e)):
            if lo == hi:
                continue
            rel = np.linalg.norm(g[lo:hi] - ref_g[lo:hi]) / np.linalg.norm(ref_g[lo:hi])
            print(f"  layer {k} {kind}: {rel:.2e}", flush=True)
            assert rel <= 2e-2, (k, kind)
