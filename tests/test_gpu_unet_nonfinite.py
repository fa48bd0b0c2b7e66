"""Values past fp16's range: a pixel whose image or block output is infinite must leave every other pixel alone, and is
itself what the plain-torch restatement makes of it (infinite or not a number), because operands that no output has (padding
channels, other rows of a strip, neighbouring positions of a patch row) take no part in it.

The restatement rounds to fp16 where the device does, so that the same values overflow; its convolutions run in torch's
plain loops (a blocked one pads channels as well). Finite outputs are held to the bar of the other forward tests, 2e-3 of
the largest of them. The infinite pixels stay away from the image's border: torch's upsampling multiplies the row past the
border with a weight of zero there."""
import copy

import pytest
import torch

from tests.test_gpu_unet import _net, _pyramid

pytestmark = pytest.mark.gpu


def _held_to_restatement(net, inputs, min_nonfinite, nan=False):
    from tests.ref_unet import unet_forward
    with torch.no_grad(), torch.backends.mkldnn.flags(enabled=False):
        want = unet_forward(copy.deepcopy(net), inputs)
        got = net.cuda().forward([t.cuda() for t in inputs]).cpu()
    finite = torch.isfinite(want)
    assert int((~finite).sum()) >= min_nonfinite and int(finite.sum()) > finite.numel() // 2
    wrong = (torch.isfinite(got) != finite).nonzero().tolist()
    assert not wrong, f"{len(wrong)} outputs, the first at {wrong[:6]}"
    assert not nan or torch.equal(got.isnan(), want.isnan())
    scale = want[finite].abs().max()
    assert (got[finite] - want[finite]).abs().max() < 2e-3 * scale


@pytest.mark.parametrize("filters,cin", [
    ([16, 32], 4),   # one pair of outputs, 32 inputs
    ([32, 32], 4),   # two pairs
    ([16, 48], 4),   # 64 inputs
    ([32, 64], 4),   # ... and two pairs
    ([16, 32], 3), ([32, 48], 8), ([48, 64], 16),
    ([48, 64], 4),   # the 1x1 in a kernel of its own
])
def test_an_output_past_the_range_stays_at_its_pixel(filters, cin):
    """One pixel's block output overflows; its image, and with it every operand of its neighbours, is finite."""
    net = _net(filters, 2, seed=90 + cin, cin=cin)
    w, h = 70, 37
    inputs = [0.5 * t for t in _pyramid(w, h, 2, cin, batch=2, seed=91)]
    with torch.no_grad():
        net.up1.convolution.feature_conv.weight[:, 0].mul_(0.1)
        net.up1.convolution.feature_conv.weight[1, 0, 1, 1] = 16.0
        net.up1.convolution.mask_conv.weight[1, 0] = 0.0
    for (b, y, x) in ((0, 5, 20), (1, 18, 41), (1, 31, 66)):
        inputs[0][b, 0, y, x] = 5e4
    _held_to_restatement(net, inputs, 3 * 3)


def _gates_that_take_infinities(net):
    """Every sum of an infinite channel 0 is -inf in the features (elu: -1) and +inf in the masks (sigmoid: 1)."""
    with torch.no_grad():
        for i in range(net.params.num_layers):
            b, C = net.block(i), net.params.num_input_channels
            for c in (0, C) if i < net.params.num_layers - 1 else (0,):
                b.feature_conv.weight[:, c] = -b.feature_conv.weight[:, c].abs() - 1e-3
                b.mask_conv.weight[:, c] = b.mask_conv.weight[:, c].abs() + 1e-3


@pytest.mark.parametrize("level,filters,cin", [
    (0, [16, 32], 4), (0, [32, 32], 4), (0, [16, 48], 4), (0, [16, 32], 3), (0, [32, 48], 8), (0, [48, 64], 4),
    # the coarser level's rows end with positions that no output has: 12 outputs behind 8 positions of image
    (1, [16, 20], 4), (1, [16, 40], 4), (1, [48, 28], 4),
])
def test_padding_channels_take_no_part(level, filters, cin):
    """An infinite image channel that the gates turn into finite outputs: of the padding channels, whose weights are zero,
    nothing comes out either."""
    net = _net(filters, 2, seed=100 + cin, cin=cin)
    _gates_that_take_infinities(net)
    inputs = _pyramid(70, 38, 2, cin, batch=2, seed=101)
    for (b, y, x) in ((0, 5, 8), (1, 9, 17), (1, 15, 32)):
        inputs[level][b, 0, y, x] = 1e5  # (infinite as an operand)
    # the infinite image reaches the output through the 1x1, at its own pixel
    _held_to_restatement(net, inputs, 3 * 3 if level == 0 else 0)


@pytest.mark.parametrize("level,filters,cin", [
    (0, [16, 32], 4), (0, [32, 32], 4), (0, [16, 32], 3), (0, [12, 20], 1), (0, [32, 48], 8), (0, [48, 64], 16), (0, [48, 64], 4),
    # behind the image, a row of the patch holds the upsampled one
    (1, [16, 20], 3), (1, [24, 20], 6), (1, [32, 36], 8), (1, [40, 56], 12), (1, [48, 64], 16),
])
def test_the_output_convolution_reads_the_image_alone(level, filters, cin):
    """The 1x1's products over the image: an infinite channel gives what its weight makes of it, and of what lies beside the
    image in the same row nothing comes out."""
    net = _net(filters, 2, seed=110 + cin, cin=cin)
    _gates_that_take_infinities(net)
    inputs = _pyramid(70, 38, 2, cin, batch=2, seed=111)
    for (b, y, x) in ((0, 5, 8), (1, 9, 17), (1, 15, 32)):
        inputs[level][b, 0, y, x] = 1e5
    _held_to_restatement(net, inputs, 3 * 3 if level == 0 else 0, nan=True)
