"""The shape kernels at the edges of their tiles (64-vertex chunks, 16 subjects, blocks of 8 and tiles of
16 basis rows) against the same model in float64.  Tolerances: float32 sums of K (forward) and of 3N
(gradients) terms, sqrt(n) roundings of 6e-8 on the size of the summed terms, with a factor of 8."""
import pytest
import torch

from gvv_amd import fit

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,N,K", [(1, 1, 1), (3, 63, 7), (4, 64, 8), (5, 65, 9), (16, 129, 16), (17, 200, 17), (33, 1000, 127),
                                   (2, 777, 128), (70, 64, 80)])
def test_shape_tiles(device, B, N, K):
    g = torch.Generator().manual_seed(B * 1000 + N + K)
    r = lambda *s: torch.randn(s, generator=g)
    alpha, pose, templ, basis, centre, gv = r(B, K), 0.3 * r(B, 6), 100 * r(N, 3), 5 * r(K, 3 * N), r(3), r(B, N, 3)
    a, p = alpha.to(device).requires_grad_(True), pose.to(device).requires_grad_(True)
    v = fit.ShapeVertices.apply(a, p, templ.to(device), basis.to(device), centre.to(device))
    ga, gp = torch.autograd.grad(v, [a, p], grad_outputs=gv.to(device))
    a64, p64 = alpha.double().requires_grad_(True), pose.double().requires_grad_(True)
    X = templ.double() - centre.double() + (a64 @ basis.double()).view(B, N, 3)
    R = fit.rodrigues(p64[:, :3])
    v64 = X @ R.transpose(1, 2) + centre.double() + 100.0 * p64[:, None, 3:]
    ga64, gp64 = torch.autograd.grad(v64, [a64, p64], grad_outputs=gv.double())
    eps = 8 * 6e-8
    size_v = float(X.abs().max()) + 100.0 * float(p64.abs().max()) + 5.0 * K ** 0.5 * float(alpha.abs().max())
    assert float((v.cpu().double() - v64).abs().max()) <= eps * K ** 0.5 * size_v
    size_a = 5.0 * 4 * float(gv.abs().max()) * (3 * N) ** 0.5
    assert float((ga.cpu().double() - ga64).abs().max()) <= eps * (3 * N) ** 0.5 * size_a
    size_p = 3.0 * (size_v + 100.0) * float(gv.abs().max()) * (3 * N) ** 0.5
    assert float((gp.cpu().double() - gp64).abs().max()) <= eps * (3 * N) ** 0.5 * size_p
