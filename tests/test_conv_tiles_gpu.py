"""The network's MFMA convolutions at the edges of their tiles (16 channels,
16 positions or 16 (channel, tap) columns, 4 deep) against torch in float64.

Tolerance: every output is a float32 sum of n products, whose error is at
most n * 2^-24 * sum |terms|; the products' sums of absolute values come from
the same convolutions on absolute values."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,cin,cout,B", [(8, 8, 32, 32, 5), (1, 1, 1, 1, 1), (2, 3, 1, 4, 3), (3, 5, 5, 17, 2),
                                           (7, 9, 16, 33, 257), (4, 4, 33, 16, 4), (10, 10, 24, 24, 1),
                                           (32, 32, 3, 32, 2), (5, 6, 64, 28, 3), (9, 2, 28, 64, 300)])
def test_conv_layer_matches_float64(H, W, cin, cout, B):
    import ctypes

    from tnsp_amd import _lib

    lib, check = _lib.lib(), _lib.check
    g = torch.Generator().manual_seed(H * 1000 + W * 100 + cin + cout)
    x, dy = torch.randn(B, cin, H, W, generator=g), torch.randn(B, cout, H, W, generator=g)
    w, bias = torch.randn(cout, cin, 3, 3, generator=g).bfloat16(), torch.randn(cout, generator=g)
    d = [t.cuda().contiguous() for t in (x, dy, w.view(torch.int16), bias)]
    p = [ctypes.c_void_p(t.data_ptr()) for t in d]
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    y, dx = torch.full((B, cout, H, W), np.nan, device="cuda"), torch.full((B, cin, H, W), np.nan, device="cuda")
    dw, db = torch.full((cout, cin, 3, 3), np.nan, device="cuda"), torch.full((cout,), np.nan, device="cuda")
    q = [ctypes.c_void_p(t.data_ptr()) for t in (y, dx, dw, db)]
    check(lib.tns_conv3x3_forward(p[0], p[2], p[3], q[0], B, cin, cout, H, W, 1, st))
    check(lib.tns_conv3x3_backward_data(p[1], q[0], p[2], q[1], B, cin, cout, H, W, st))
    ws = ctypes.c_int64()
    check(lib.tns_conv3x3_backward_weight_workspace(B, cin, cout, ctypes.byref(ws)))
    work = torch.empty(ws.value // 4, device="cuda")
    check(lib.tns_conv3x3_backward_weight(p[1], q[0], p[0], q[2], q[3], B, cin, cout, H, W,
                                          ctypes.c_void_p(work.data_ptr()), st))
    torch.cuda.synchronize()
    eps = 2.0 ** -24
    X, DY, Wt, Bi = x.double(), dy.double(), w.double(), bias.double()
    ref = F.conv2d(X, Wt, Bi, padding=1).relu()
    n = 9 * cin + 2
    tol = n * eps * F.conv2d(X.abs(), Wt.abs(), Bi.abs(), padding=1)
    assert torch.all((y.cpu().double() - ref).abs() <= tol)
    G = torch.where(y.cpu() > 0, DY, 0.0)  # the layer's own ReLU mask
    ref = F.conv_transpose2d(G, Wt, padding=1)
    assert torch.all((dx.cpu().double() - ref).abs() <= 9 * cout * eps * F.conv_transpose2d(G.abs(), Wt.abs(), padding=1) + 1e-30)

    def grad_w(a, b):
        return F.conv2d(a.transpose(0, 1), b.transpose(0, 1), padding=1).transpose(0, 1)

    n = B * H * W
    assert torch.all((dw.cpu().double() - grad_w(X, G)).abs() <= n * eps * grad_w(X.abs(), G.abs()) + 1e-30)
    assert torch.all((db.cpu().double() - G.sum((0, 2, 3))).abs() <= n * eps * G.abs().sum((0, 2, 3)) + 1e-30)


def test_layer_beyond_lds_is_refused():
    """64 channels of 32 x 32: the padded planes exceed a CU's 160 KB."""
    from tnsp_amd import _lib

    t = torch.zeros(2 * 64 * 34 * 34, device="cuda")
    p = t.data_ptr()
    with pytest.raises(RuntimeError, match="exceeds LDS"):
        _lib.check(_lib.lib().tns_conv3x3_backward_data(p, p, p, p, 2, 3, 64, 32, 32,
                                                        torch.cuda.current_stream().cuda_stream))


@pytest.mark.parametrize("v", [1.1454734802246094, 1.1126136779785156, 1.8636400699615479])
def test_partial_gradients_add_in_short_chains(v):
    """1024 equal samples, whose sums round one way in a long chain: two
    additions within a workgroup, then 16 + 3 + 2 over the 512 workgroups, each
    off by at most 2^-24 of the sum."""
    import ctypes

    from tnsp_amd import _lib

    lib, check = _lib.lib(), _lib.check
    B = 1024
    x, dy = torch.ones(B, device="cuda"), torch.full((B,), v, device="cuda")
    dw, db = torch.empty(9, device="cuda"), torch.empty(1, device="cuda")
    ws = ctypes.c_int64()
    check(lib.tns_conv3x3_backward_weight_workspace(B, 1, 1, ctypes.byref(ws)))
    work = torch.empty(ws.value // 4, device="cuda")
    check(lib.tns_conv3x3_backward_weight(dy.data_ptr(), None, x.data_ptr(), dw.data_ptr(), db.data_ptr(), B, 1, 1, 1,
                                          1, work.data_ptr(), torch.cuda.current_stream().cuda_stream))
    exact = B * float(dy[0].cpu())
    for got in (float(dw[4]), float(db[0])):
        assert abs(got - exact) <= 23 * 2.0 ** -24 * exact
