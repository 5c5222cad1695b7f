"""The 3x3 weight gradient of rows of whole 4-pixel runs at the edges of its
tiles: channel counts around 32, images of one and several blocks of 64 pixels
and ragged last ones, runs across rows and images, and next to them the shapes
that stay with the general kernel (few pixels, other widths), against the bf16
oracle at the tolerance of single convolutions; and a network whose levels take
both kernels in one gradient."""
import pytest

import test_gpu_unet as layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("relu", [False, True])
@pytest.mark.parametrize("n,cin,cout,h,w", [
    (8, 1, 1, 4, 4), (2, 31, 33, 16, 4), (5, 33, 32, 7, 12), (1, 32, 65, 1, 128), (3, 64, 31, 9, 20),
    (1, 5, 70, 33, 64), (2, 96, 8, 3, 100), (17, 34, 3, 2, 8), (1, 8, 8, 3, 40), (2, 8, 8, 12, 14),
])
def test_weight_gradient_edges(ctx, relu, n, cin, cout, h, w):
    layer.test_conv_layer_matches_oracle(ctx, 2, relu, n, cin, cout, h, w, 3)


@pytest.mark.parametrize("levels,base,n,hw", [(3, 8, 3, 24), (4, 4, 2, 40)])
def test_mixed_levels_gradient(ctx, levels, base, n, hw):
    layer.test_gradient_matches_oracle(ctx, levels, base, n, hw)
