"""The bf16 copies of the weights at the edges of their 32 x 64 tiles, several layers to a launch and
with and without the transpose: equal to torch's rounding, bit for bit, nothing written beyond them."""
import ctypes

import pytest
import torch

from gvv_amd import _lib

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (32, 9, 8), (33, 9, 8), (31, 1, 63), (32, 1, 64), (64, 1, 65), (5, 9, 3), (63, 4, 16), (7, 25, 1),
          (128, 1, 4096), (65, 9, 129), (2, 3, 7), (256, 9, 64), (3, 1, 1), (1, 9, 256), (34, 2, 33), (96, 1, 128), (1, 1, 200)]


@pytest.mark.parametrize("layers", [[s] for s in SHAPES] + [SHAPES], ids=lambda s: str(s[0]) if len(s) == 1 else "all")
def test_prepared_weights(device, layers):
    g = torch.Generator().manual_seed(len(layers) + layers[0][0])
    w = [torch.randn(s, generator=g).to(device) for s in layers]
    pad = 64
    wb = [torch.full((x.numel() + pad,), -7.0, dtype=torch.bfloat16, device=device) for x in w]
    wt = [torch.full((x.numel() + pad,), -7.0, dtype=torch.bfloat16, device=device) for x in w]
    bare = [len(w) > 1 and k % 5 == 4 for k in range(len(w))]       # no transpose asked for
    n = len(w)
    ints, ptrs = ctypes.c_int32 * n, ctypes.c_void_p * n
    stream = torch.cuda.current_stream().cuda_stream
    _lib.check(_lib.load().gvv_conv_prepare_weights_layers(
        n, ints(*(s[0] for s in layers)), ints(*(s[1] for s in layers)), ints(*(s[2] for s in layers)),
        ptrs(*(x.data_ptr() for x in w)), ptrs(*(x.data_ptr() for x in wb)),
        ptrs(*(None if b else x.data_ptr() for x, b in zip(wt, bare))), stream), "gvv_conv_prepare_weights_layers")
    for x, b, t, no in zip(w, wb, wt, bare):
        h = x.to(torch.bfloat16)
        assert torch.equal(b[:-pad], h.reshape(-1)) and bool((b[-pad:] == -7).all())
        if no:
            assert bool((t == -7).all())
        else:
            assert torch.equal(t[:-pad], h.permute(2, 1, 0).reshape(-1)) and bool((t[-pad:] == -7).all())
