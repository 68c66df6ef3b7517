"""The convolution kernels with enough pixels for the 64 x 128 tiles (1024 of them) and with 64 x 64 tiles of
two waves, at ragged sizes, against the FP64 conv oracle with test_gpu_conv's bounds."""
import numpy as np
import pytest
import torch

from gvv_amd import _lib
from oracle import conv_oracle as CO
from test_gpu_conv import P, S, bf, check_close, rnd

pytestmark = pytest.mark.gpu

GEOMS = [
    # B, H, W, Cin, Cout, ks, stride, pad
    (2, 257, 256, 64, 40, 3, 1, 1),       # forward: 1,028 tiles of 64 x 128, partial in both directions
    (1, 363, 362, 48, 520, 1, 1, 0),      # backward data the same (17 steps)
    (3, 75, 77, 40, 72, 3, 1, 1),         # two waves, 12 steps: two rounds of loads
    (9, 43, 43, 64, 96, 3, 1, 1),         # two waves, 18 steps: three rounds
    (5, 64, 64, 72, 64, 3, 2, 1),         # two waves in the residue classes
]


@pytest.mark.parametrize("geom", GEOMS, ids=lambda g: "x".join(map(str, g)))
def test_conv_wide(device, geom):
    B, H, W, Cin, Cout, ks, st, pad = geom
    L = _lib.load()
    rng = np.random.default_rng(sum(v * 7 ** i for i, v in enumerate(geom)))
    OH, OW = CO.out_size(H, ks, st, pad), CO.out_size(W, ks, st, pad)
    x, w = rnd(rng, (B, H, W, Cin)), rnd(rng, (Cout, ks, ks, Cin), 1.0 / np.sqrt(ks * ks * Cin))
    b, dz = rng.standard_normal(Cout).astype(np.float32) * 0.1, rnd(rng, (B, OH, OW, Cout))
    xd, dzd, bd, wf = bf(x, device), bf(dz, device), torch.from_numpy(b).to(device), torch.from_numpy(w).to(device)
    wb = torch.empty(w.shape, dtype=torch.bfloat16, device=device)
    wt = torch.empty((Cin, ks, ks, Cout), dtype=torch.bfloat16, device=device)
    _lib.check(L.gvv_conv_prepare_weights(Cout, ks * ks, Cin, P(wf), P(wb), P(wt), S()), "prepare")
    y = torch.full((B, OH, OW, Cout), 7.0, device=device)
    dx = torch.full((B, H, W, Cin), 7.0, dtype=torch.bfloat16, device=device)
    _lib.check(L.gvv_conv_forward(*geom, P(xd), P(wb), P(bd), 0, P(y), 1, S()), "fwd")
    _lib.check(L.gvv_conv_backward_data(*geom, P(dzd), P(wt), P(xd), P(dx), S()), "bwd data")
    check_close("forward", y.cpu().numpy(), CO.conv_forward(x, w, b, st, pad), CO.conv_abs_bound(x, w, st, pad) + np.abs(b), False)
    rdx, bdx = CO.conv_backward(x, w, dz, st, pad)[0], CO.conv_backward_abs_bound(x, w, dz, st, pad)[0]
    check_close("backward data", dx.float().cpu().numpy(), rdx * (x > 0), bdx, True)
