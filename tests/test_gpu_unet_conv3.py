"""The packed 3x3 kernel at the edges of its tiles: channel counts around its
16-channel steps and 32-row tiles, images around its 4x8, 8x8 and 8x16 pixel
tiles, every dispatch (1, 2-3 and more row tiles), against the bf16 oracle at
the tolerance of single convolutions (FP32 accumulation order, 2e-5)."""
import pytest

import test_gpu_unet as layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n,cin,cout,h,w", [
    (1, 1, 1, 1, 2), (1, 16, 31, 3, 5), (2, 17, 33, 4, 8), (1, 33, 97, 5, 9), (3, 15, 128, 8, 8),
    (1, 48, 129, 2, 31), (2, 9, 64, 17, 16), (1, 32, 32, 16, 33),
])
def test_packed_conv_edges(ctx, mode, n, cin, cout, h, w):
    layer.test_conv_layer_matches_oracle(ctx, mode, True, n, cin, cout, h, w, 3)
