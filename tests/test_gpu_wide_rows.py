"""Linears whose output rows are so long that 32 of them pass 4 GiB: the epilogue's
32-bit offsets do not reach, and the launch takes the kernels that store with 64."""
import pytest
import torch

import gsplat_hip as G
from gpu_util import case, stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flags,tol", [(0, 1e-5), (G.EPI_BF16, 2e-2), (G.EPI_F32X6, 1e-5)])
def test_linear_of_wide_rows(flags, tol):
    case(f"wide rows {flags}")
    M, K, N = 40, 32, 34_700_032
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.empty(M, K, device="cuda").normal_(generator=g)
    w = torch.empty(N, K, device="cuda").normal_(generator=g)
    y = torch.zeros(M, N, device="cuda")
    G.check(G.lib().gs_hip_linear(G.ptr(x), G.ptr(w), None, G.ptr(y), M, K, N, 0, flags, None, stream()))
    torch.cuda.synchronize()
    for at in (0, N // 2, N - 512):
        ref = x.double() @ w[at:at + 512].double().t()
        assert (y[:, at:at + 512] - ref).abs().max() <= tol * 10


@pytest.mark.parametrize("H,W,k,s,p", [(3, 1, 3, 1, 1), (7, 5, 3, 2, 1), (2, 300, 5, 1, 2), (40, 3, 3, 1, 0), (16, 16, 3, 1, 2)])
def test_conv_windows_over_image_borders(H, W, k, s, p):
    """Tiles of 128 output pixels that span many small images, and a padding wider
    than half the window."""
    case(f"conv borders {H}x{W} k={k} s={s} p={p}")
    Ci, Co = 128, 256
    Ho, Wo = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    B = max(2, 5000 // (Ho * Wo))
    g = torch.Generator(device="cuda").manual_seed(2)
    x = torch.empty(B, H, W, Ci, device="cuda").normal_(generator=g)
    w = torch.empty(Co, k, k, Ci, device="cuda").normal_(generator=g)
    y = torch.zeros(B, Ho, Wo, Co, device="cuda")
    G.check(G.lib().gs_hip_conv2d(G.ptr(x), B, H, W, Ci, G.ptr(w), None, G.ptr(y), Co, k, s, p, 1, 0, None, stream()))
    torch.cuda.synchronize()
    ref = torch.nn.functional.conv2d(x.cpu().double().permute(0, 3, 1, 2), w.cpu().double().permute(0, 3, 1, 2),
                                     stride=s, padding=p).permute(0, 2, 3, 1)
    assert (y.cpu() - ref).abs().max() <= 2e-5 * (k * k * Ci) ** 0.5
