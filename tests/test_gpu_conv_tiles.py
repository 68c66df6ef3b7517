"""The convolution kernels at the edges of their tiles and stretches, against the FP64 conv oracle
with test_gpu_conv's bounds: channel counts on both sides of 16, 32 and 64 and off the multiple of
32, pixel counts around tile sizes and rows shorter than 8, reductions of one step, one stretch and
several, strides with empty residue classes, and outputs that are not 16-byte aligned."""
import ctypes

import numpy as np
import pytest
import torch

from gvv_amd import _lib
from oracle import conv_oracle as CO
from test_gpu_conv import P, S, bf, check_close, rnd

pytestmark = pytest.mark.gpu

GEOMS = [
    # B, H, W, Cin, Cout, ks, stride, pad
    (1, 1, 1, 8, 8, 1, 1, 0),           # one pixel, one chunk
    (17, 1, 1, 264, 40, 1, 1, 0),       # 33 chunks: a partial last step
    (3, 5, 13, 40, 72, 3, 2, 1),        # nothing a multiple of a tile
    (2, 12, 12, 64, 64, 3, 3, 0),       # stride 3
    (2, 4, 7, 32, 16, 1, 3, 0),         # classes without taps: zeros
    (1, 34, 36, 96, 48, 3, 2, 1),
    (4, 128, 128, 8, 32, 3, 2, 1),      # one wave per tile, three steps
    (2, 128, 160, 32, 64, 3, 2, 1),     # one wave per tile
    (16, 32, 32, 64, 128, 3, 2, 1),     # 64 x 64 tiles, several waves
    (2, 6, 6, 512, 24, 3, 1, 1),        # a reduction of 144 steps
]


@pytest.mark.parametrize("geom", GEOMS, ids=lambda g: "x".join(map(str, g)))
def test_conv_tiles(device, geom):
    B, H, W, Cin, Cout, ks, st, pad = geom
    L = _lib.load()
    rng = np.random.default_rng(sum(v * 7 ** i for i, v in enumerate(geom)))
    OH, OW = CO.out_size(H, ks, st, pad), CO.out_size(W, ks, st, pad)
    x, w = rnd(rng, (B, H, W, Cin)), rnd(rng, (Cout, ks, ks, Cin), 1.0 / np.sqrt(ks * ks * Cin))
    b, dz = rng.standard_normal(Cout).astype(np.float32) * 0.1, rnd(rng, (B, OH, OW, Cout))
    xd, dzd, bd = bf(x, device), bf(dz, device), torch.from_numpy(b).to(device)
    wf = torch.from_numpy(w).to(device)
    wb = torch.empty(w.shape, dtype=torch.bfloat16, device=device)
    wt = torch.empty((Cin, ks, ks, Cout), dtype=torch.bfloat16, device=device)
    _lib.check(L.gvv_conv_prepare_weights(Cout, ks * ks, Cin, P(wf), P(wb), P(wt), S()), "prepare")
    ref, bound = CO.conv_forward(x, w, b, st, pad), CO.conv_abs_bound(x, w, st, pad) + np.abs(b)
    rdx, rdw, rdb = CO.conv_backward(x, w, dz, st, pad)
    bdx, bdw, bdb = CO.conv_backward_abs_bound(x, w, dz, st, pad)
    g = (B, H, W, Cin, Cout, ks, st, pad)
    for shift in (0, 1):           # shift 1: outputs off 16-byte alignment
        def out(shape, dtype):
            n = int(np.prod(shape))
            return torch.full((n + 8,), 7.0, dtype=dtype, device=device)[shift:shift + n].view(shape)
        yf, y = out((B, OH, OW, Cout), torch.float32), out((B, OH, OW, Cout), torch.bfloat16)
        _lib.check(L.gvv_conv_forward(*g, P(xd), P(wb), P(bd), 0, P(yf), 1, S()), "fwd f32")
        _lib.check(L.gvv_conv_forward(*g, P(xd), P(wb), P(bd), 1, P(y), 0, S()), "fwd")
        check_close("forward f32", yf.cpu().numpy(), ref, bound, False)
        check_close("forward relu bf16", y.float().cpu().numpy(), np.maximum(ref, 0.0), bound, True)
        dx = out((B, H, W, Cin), torch.bfloat16)
        _lib.check(L.gvv_conv_backward_data(*g, P(dzd), P(wt), P(xd), P(dx), S()), "bwd data")
        check_close("backward data", dx.float().cpu().numpy(), rdx * (x > 0), bdx, True)
        ws = torch.empty(int(L.gvv_conv_workspace_floats(*g)), device=device)
        dw, db = out((Cout, ks, ks, Cin), torch.float32), out((Cout,), torch.float32)
        _lib.check(L.gvv_conv_backward_weight(*g, P(xd), P(dzd), P(dw), P(db), P(ws), ws.numel(), S()), "bwd weight")
        check_close("backward weight", dw.cpu().numpy(), rdw, bdw, False)
        check_close("backward bias", db.cpu().numpy(), rdb, bdb, False)


def test_prepare_weights_layers(device):
    """Several layers in one launch (more than one launch's 16) equal the layers one by one."""
    L = _lib.load()
    sizes = [(8 * (1 + i % 5), (1, 4, 9)[i % 3], 8 * (1 + i % 7)) for i in range(18)]
    g = torch.Generator().manual_seed(1)
    ws = [torch.randn(s, generator=g).to(device) for s in sizes]
    wb = [torch.zeros(s, dtype=torch.bfloat16, device=device) for s in sizes]
    wt = [torch.zeros((s[2], s[1], s[0]), dtype=torch.bfloat16, device=device) for s in sizes]
    n = len(sizes)
    ints, ptrs = ctypes.c_int32 * n, ctypes.c_void_p * n
    wt_ptrs = [t.data_ptr() for t in wt]
    wt_ptrs[3] = None
    _lib.check(L.gvv_conv_prepare_weights_layers(n, *(ints(*(s[k] for s in sizes)) for k in range(3)),
                                                 ptrs(*(t.data_ptr() for t in ws)), ptrs(*(t.data_ptr() for t in wb)),
                                                 ptrs(*wt_ptrs), S()), "layers")
    for i, w in enumerate(ws):
        assert torch.equal(wb[i], w.to(torch.bfloat16))
        assert torch.equal(wt[i], torch.zeros_like(wt[i]) if i == 3 else w.to(torch.bfloat16).permute(2, 1, 0).contiguous())
