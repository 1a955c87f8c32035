"""Convolutions and weight gradients of tiles staged in LDS (k_conv_tile,
k_wgrad_tile) against the float32 oracle: images narrower and lower than a tile, with one pixel left over, with
uneven halves under the upsampled input, tiles limited by the LDS (deep
channels, dilated bottlenecks) and images whose bottleneck fits no tile.  The
bars are those of the network's BF16 arithmetic: 3e-2 of the output, 1e-1 of
each layer's gradient, a cosine above 0.99."""
import numpy as np
import pytest

import parallellbmcranfield_amd as lbm
from oracle import nn_oracle as NN
from test_gpu_nn import _rel, _sample

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,levels,dil", [(2, 9, 2, 1), (9, 2, 2, 1), (5, 64, 2, 1),
                                            (17, 65, 3, 1), (66, 16, 3, 2), (21, 130, 4, 3),
                                            (40, 41, 4, 4), (33, 34, 2, 9), (50, 45, 2, 16)])
def test_tiles_match_oracle(H, W, levels, dil):
    print("conv tiles", H, W, levels, dil, flush=True)
    net = lbm.Net(H, W, batch=3, base=32, levels=levels, seed=6, in_channels=4, dilation=dil)
    p = net.params()
    inp, tgt = _sample(3, H, W, 5, 4)
    y = net.predict(inp)
    assert _rel(y, NN.forward(p, inp, levels, 32, dil=dil)) < 3e-2
    loss, g = net.gradients(inp, tgt)
    loss_ref, g_ref = NN.loss_and_grad(p, inp, tgt, levels, 32, dil)
    assert abs(loss - loss_ref) <= 3e-2 * loss_ref
    for (w, b), (wr, br) in zip(NN.unpack(g, levels, 32)[0], NN.unpack(g_ref, levels, 32)[0]):
        cos = float((w * wr).sum() / (np.linalg.norm(w) * np.linalg.norm(wr) + 1e-30))
        assert _rel(w, wr) < 1e-1 and cos > 0.99 and _rel(b, br) < 1e-1
    assert np.isfinite(net.gradients(inp[:1], tgt[:1])[1]).all()  # fewer, other chunks
    net.close()
