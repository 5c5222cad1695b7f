"""Single 3x3 convolutions at the channel count from which their weights are
packed (8 reduction channels), against the oracle with the tolerance of the layer
test."""
import pytest

import test_gpu_unet as layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("cin,cout", [(7, 8), (8, 7), (8, 8), (1, 9)])
def test_edges_of_the_rule(ctx, mode, cin, cout):
    layer.test_conv_layer_matches_oracle(ctx, mode, True, 2, cin, cout, 9, 12, 3)
