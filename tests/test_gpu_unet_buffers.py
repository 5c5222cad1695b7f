"""Buffers that the surrogate's device entry points do not work on in place:
pinned host memory and addresses off the element size are copied, and give
the bits of an ordinary device tensor."""
import ctypes as C

import numpy as np
import pytest

import multislice_amd as msx

pytestmark = pytest.mark.gpu

DEVICE = 1


def ptr(t):
    return C.c_void_p(t.data_ptr())


def pinned(t):
    import torch
    p = torch.empty(t.shape, dtype=t.dtype, pin_memory=True)
    p.copy_(t)
    return p


def shifted(t):
    """The tensor's bytes two past an aligned address."""
    import torch
    raw = torch.empty(t.numel() * 4 + 16, dtype=torch.uint8, device="cuda")
    raw[2:2 + t.numel() * 4] = t.reshape(-1).view(torch.uint8)
    return raw[2:2 + t.numel() * 4]


@pytest.mark.parametrize("place", [pinned, shifted])
@pytest.mark.parametrize("cin", [1, 3])
def test_other_buffers_give_the_same_bits(ctx, cin, place):
    import torch
    L = msx.load()
    n, h, w = 2, 16, 24
    g = torch.Generator(device="cuda").manual_seed(cin)
    x = torch.rand((n, cin, h, w), generator=g, device="cuda")
    t = torch.rand((n, h, w), generator=g, device="cuda")
    nets = [msx.UNet(ctx, 3, 8, 5, in_channels=cin) for _ in range(2)]
    want = torch.empty((n, h, w), device="cuda")
    torch.cuda.synchronize()
    assert L.msx_unet_forward(nets[0].h, ptr(x), ptr(want), n, h, w, DEVICE) == 0
    px, pt, py = place(x), place(t), place(torch.zeros_like(t))
    torch.cuda.synchronize()
    assert L.msx_unet_forward(nets[1].h, ptr(px), ptr(py), n, h, w, DEVICE) == 0
    assert bytes(py.cpu().numpy().tobytes()) == want.cpu().numpy().tobytes()
    loss = [C.c_double(), C.c_double()]
    for net, a, b, out in ((nets[0], x, t, loss[0]), (nets[1], px, pt, loss[1])):
        assert L.msx_unet_train_step(net.h, ptr(a), ptr(b), n, h, w, 1e-3, C.byref(out), DEVICE) == 0
    assert loss[0].value == loss[1].value
    np.testing.assert_array_equal(nets[0].params(), nets[1].params())
    for net in nets:
        net.close()
