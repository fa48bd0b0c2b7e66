"""The net's kernels at the edges of their dispatch, against the plain-torch restatement: workgroups of one to four output
pairs on either side of the lines between them, sizes at the edges of the 8 x 32 tiles. Bars of tests/test_gpu_unet.py: 2e-3 of the largest output against the restatement that
rounds where the device rounds (summation order, fast exp), 2e-2 of each gradient's largest element (fp16 operands)."""
import copy

import numpy as np
import pytest
import torch

from tests.test_gpu_unet import GRAD_TOL, _compare, _net, _pyramid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("filters,w,h,cin,batch", [
    ([48, 64], 33, 9, 4, 1),        # 44 outputs at the finest level: three pairs, 64 inputs
    ([64, 64], 31, 7, 3, 2),        # 61: four pairs, the last one nearly empty; an odd number of image channels
    ([64, 32], 35, 12, 4, 2),       # ... on 32 inputs
    ([60, 64], 40, 11, 16, 1),      # three pairs, sixteen image channels
    ([64, 32], 64, 16, 8, 1),       # whole tiles
    ([36, 24], 65, 17, 2, 3),       # 34: the third pair holds two outputs
    ([32, 16], 160, 120, 4, 1),     # 75 and 24 tiles: a workgroup each, dealt to the eight XCDs
    ([32, 36], 40, 40, 4, 1),       # 28 outputs on 36 inputs: the block's own 1x1 with two pairs and 64 channels
    ([32, 24], 544, 272, 4, 1),     # enough tiles for two pairs per workgroup at both levels
    ([48, 64], 544, 272, 4, 1),     # ... at the coarser level only (the finest has three pairs)
    ([64, 64], 544, 136, 6, 2),
    # image channels that end inside a group of eight, with upsampled ones behind them
    ([24, 32, 32], 70, 41, 5, 2),
    ([24, 48, 40], 70, 41, 7, 2),
    ([40, 60, 56], 45, 50, 12, 1),
    # three and four pairs at the coarser levels, either side of the 512 tiles from which they share a workgroup:
    ([16, 48], 129, 65, 4, 35),     # 3 x 5 tiles x 35 images
    ([16, 48, 52], 126, 64, 4, 63), # 2 x 4 x 63: not enough
    ([16, 50, 52], 130, 64, 4, 45), # 3 x 4 x 45, 64 inputs
    ([16, 60, 56], 130, 64, 2, 45), # four pairs
    ([16, 62, 30], 130, 66, 1, 35), # ... on 32 inputs
    # the data gradient's strips, of 15 coarser columns and 4 n - 1 coarser rows:
    ([16, 32], 30, 6, 4, 1),        # one strip, filled exactly
    ([32, 32], 31, 7, 3, 2),        # a column and a row more, odd sizes, outputs that start at position 6
    ([16, 48], 60, 14, 6, 1),       # two strips; 64 inputs
    ([32, 48], 29, 5, 16, 1),       # sixteen image channels
    ([16, 32], 302, 166, 4, 4),     # strips of several steps, two workgroups per CU, the last strip a short one
    ([32, 32], 301, 203, 8, 3),     # ... one workgroup per CU, odd sizes
    ([16, 48], 301, 95, 2, 5),
    ([32, 48], 290, 131, 4, 3),     # 64 pre-activations x 64 inputs
    # the weight gradient takes 128 pre-activations on 32 inputs in one workgroup from 512 tiles on
    ([64, 32], 290, 131, 4, 3),     # 10 x 17 x 3: two short of it
    ([62, 30], 290, 129, 3, 4),
])
def test_forward_and_gradients_at_dispatch_edges(filters, w, h, cin, batch):
    _held_to_restatement(filters, w, h, cin, batch)


def _held_to_restatement(filters, w, h, cin, batch):
    from tests.ref_unet import unet_forward
    levels = len(filters)
    net = _net(filters, levels, seed=60 + w + cin, cin=cin)
    inputs = _pyramid(w, h, levels, cin, batch=batch, seed=61)
    _compare(copy.deepcopy(net), inputs)
    g = torch.Generator().manual_seed(62)
    upstream = torch.randn((batch, 3, h, w), generator=g) * 1e-3
    ref = copy.deepcopy(net)
    ins_ref = [t.clone().requires_grad_(True) for t in inputs]
    (unet_forward(ref, ins_ref, half_rounding=False) * upstream).sum().backward()
    net = net.cuda()
    ins = [t.cuda().requires_grad_(True) for t in inputs]
    (net.forward(ins) * upstream.cuda()).sum().backward()
    pairs = [(f"d inputs[{i}]", ins[i].grad, ins_ref[i].grad) for i in range(levels)]
    pairs += [(n, p.grad, q.grad) for (n, p), (_, q) in zip(net.named_parameters(), ref.named_parameters())]
    for name, got, want in pairs:
        got, want = got.cpu().numpy(), want.numpy()
        scale = np.abs(want).max()
        assert np.abs(got - want).max() < GRAD_TOL * scale, f"{name}: {np.abs(got - want).max() / scale:.3e}"


def _strip_steps(preact, inputs, cin, coarse_w, coarse_h, batch):
    """Steps of a strip of the data gradient that takes the upsampling's adjoint with it: the fewest with which all strips
    are resident at once. (Sizes in LDS: the patch, the ring of gradients, the image's share.)"""
    image = 4 if cin <= 4 else 8 if cin <= 8 else 16
    lds = 10 * 34 * (preact + 8) * 2 + 10 * 32 * (inputs + 8) * 2 + 8 * 32 * image * 4
    per_cu = 2 if lds <= 64 * 1280 and inputs == 32 else 1
    strips, steps = (coarse_w + 14) // 15 * batch, 1
    while steps < (coarse_h + 4) // 4 and strips * ((coarse_h + 4 * steps - 2) // (4 * steps - 1)) > 256 * per_cu:
        steps += 1
    return steps


@pytest.mark.parametrize("filters,preact,inputs,w,h,cin,batch", [
    ([16, 32], 32, 32, 30, 800, 4, 24),  # two workgroups per CU
    ([32, 32], 64, 32, 29, 799, 4, 24),  # ... with twice the pre-activations
    ([32, 32], 64, 32, 29, 799, 6, 15),  # ... and more than four image channels: one
    ([16, 48], 32, 64, 30, 800, 3, 15),  # block outputs that start at position 6
    ([32, 48], 64, 64, 30, 799, 4, 15),
])
def test_gradients_through_strips_of_many_steps(filters, preact, inputs, w, h, cin, batch):
    """The strips' rings of ten rows go on by eight: their first row is 0, 8, 6, 4, 2 and, in the sixth step, 0 again."""
    assert _strip_steps(preact, inputs, cin, (w + 1) // 2, (h + 1) // 2, batch) >= 6
    _held_to_restatement(filters, w, h, cin, batch)


@pytest.mark.parametrize("batch", [10, 11, 24])
def test_gradients_with_two_workgroups_on_a_cu(batch):
    """32 inputs and 64 pre-activations, two levels of 100 and 50 tiles an image: 1500 and 1650 tiles, of which 512 workgroups of the
    weight gradient get three each from 1536 on; 24 images leave the 512 strips of the data gradient six steps, after which their
    rings are back at row 0."""
    _held_to_restatement([32, 32], 30, 800, 4, batch)


@pytest.mark.parametrize("cin,batch", [(3, 10), (3, 11), (6, 10), (6, 11), (8, 15), (8, 16), (10, 15), (10, 16), (16, 31)])
def test_weight_gradients_of_one_and_of_two_workgroups_on_a_cu(cin, batch):
    """32 inputs and 64 pre-activations for each kind of image: two workgroups on a CU from 1536 tiles on and up to eight channels.
    An image has 100 tiles and, up to six channels, 50 of the second level in the same launch; sixteen channels leave 32 inputs to
    the second level only."""
    _held_to_restatement([48, 64] if cin == 16 else [32, 32], 30, 800, cin, batch)


@pytest.mark.parametrize("filters,w,h,cin,batch", [
    ([16, 32], 37, 29, 4, 2), ([24, 32], 40, 24, 3, 1), ([32, 48], 33, 17, 8, 1), ([48, 64], 32, 8, 16, 1), ([16, 32], 1, 1, 4, 1),
])
def test_channels_last_pyramids_are_read_in_place(filters, w, h, cin, batch):
    """Views of [B, H, W, C] images (what the splat's eval mode returns) give the bits of their contiguous copies."""
    net = _net(filters, 2, seed=70 + cin, cin=cin).cuda()
    inputs = [t.cuda() for t in _pyramid(w, h, 2, cin, batch=batch, seed=71)]
    with torch.no_grad():
        want = net.forward(inputs)
        got = net.forward([t.permute(0, 2, 3, 1).contiguous().permute(0, 3, 1, 2) for t in inputs])
        mixed = net.forward([inputs[0], inputs[1].permute(0, 2, 3, 1).contiguous().permute(0, 3, 1, 2)])
    assert torch.equal(got, want) and torch.equal(mixed, want)


def test_upsampling_of_neighbours_far_apart():
    """Images near the ends of fp16's range with changing signs: their bilinear mixes stay inside it, so the net's output
    is the restatement's (a difference of two neighbours would not be: it is an infinity in fp16). Weights of 1e-4 keep
    the convolutions' sums, up to 72 x 6e4 x 1e-4, in range as well; the bar is that of the other forward tests."""
    net = _net([16, 32], 2, seed=80)
    with torch.no_grad():
        for m in net.modules():
            if isinstance(m, torch.nn.Conv2d) and m.kernel_size == (3, 3):
                m.weight.mul_(1e-4 / m.weight.abs().max())
    g = torch.Generator().manual_seed(81)
    inputs = [torch.sign(torch.rand(t.shape, generator=g) - 0.5) * (4e4 + 2e4 * t) for t in _pyramid(45, 37, 2, 4, batch=1, seed=82)]
    _compare(net, inputs)


@pytest.mark.parametrize("filters,w,h,batch", [
    ([32, 32, 32, 32, 32], 160, 120, 1),  # one instance for all levels, a workgroup per tile
    ([32, 32, 32, 32], 545, 273, 2),      # ... more tiles than workgroups
    ([16, 32, 48, 64], 300, 200, 2),      # levels of several instances, two of which share one, a level of two shares
])
def test_weight_gradients_of_some_levels(filters, w, h, batch):
    """Levels whose weight gradients are the same instance of the kernel run in one launch, whose workgroups are dealt to the
    levels that are asked for: without the gradients of some levels (weights, biases or both), the others are those that all
    of them together give, the same bits where the tiles are dealt alike."""
    import ctypes as C

    from trips_amd import _lib, abi
    from trips_amd.renderer import get_context
    from trips_amd.unet import _buffer_sizes, _ptr, _stream_ptr
    L = len(filters)
    net = _net(filters, L, seed=5).cuda()
    ins = [t.cuda() for t in _pyramid(w, h, L, 4, batch=batch, seed=6)]
    ctx, dev, d, params = get_context(0), ins[0].device, net.desc(ins), net.ordered_parameters()
    sizes = _buffer_sizes(bytes(d))
    saved, ws = ctx.alloc_bytes(sizes[1]), ctx.alloc_bytes(sizes[2])
    with torch.no_grad():
        net._run_forward(d, ins, params, saved)
    d_out = torch.randn((batch, 3, h, w), generator=torch.Generator().manual_seed(7)).cuda() * 1e-3
    wts, _ = net._weights_struct(params)

    def backward(wanted):
        """wanted: (weights, biases) per level"""
        outs = [torch.full_like(p, float("nan")) for p in params]
        g, d_ins = abi.TripsUnetGrads(), [torch.empty_like(t) for t in ins]
        for i, (weights, biases) in enumerate(wanted):
            f, fb, m, mb = (t.data_ptr() for t in outs[4 * i:4 * i + 4])
            g.feature_weight[i], g.mask_weight[i] = (f, m) if weights else (None, None)
            g.feature_bias[i], g.mask_bias[i] = (fb, mb) if biases else (None, None)
        g.inputs[:L] = [t.data_ptr() for t in d_ins]
        _lib.check(ctx.lib.trips_unet_backward(ctx.ctx, C.byref(d), C.byref(wts), net._input_ptrs(ins), _ptr(saved), _ptr(d_out),
                                               C.c_float(net.grad_scale), C.byref(g), _ptr(ws), sizes[2], _stream_ptr(dev)))
        return outs, d_ins
    full, full_ins = backward([(True, True)] * L)
    assert all(bool(torch.isfinite(t).all()) for t in full[:4 * L])
    # 8 x 32 tiles, at most two shares of each: up to 240 of them find a workgroup of their own whatever is asked for
    few = 2 * batch * sum(-(-t.shape[2] // 8) * -(-t.shape[3] // 32) for t in ins) <= 240
    for wanted in ([(i != 1, True) for i in range(L)], [(True, i != 0) for i in range(L)], [(i % 2 == 0, i < 2) for i in range(L)],
                   [(i == L - 1, False) for i in range(L)]):
        part, part_ins = backward(wanted)
        assert all(torch.equal(a, b) for a, b in zip(part_ins, full_ins))
        dealt_alike = few or all(weights for weights, _ in wanted)
        for i, (weights, biases) in enumerate(wanted):
            for k in range(4):
                a, b = part[4 * i + k], full[4 * i + k]
                if not (weights if k % 2 == 0 else biases):
                    assert bool(torch.isnan(a).all())
                elif k % 2 == 1 and not weights:  # summed by a kernel of its own: single precision, another order
                    assert float((a - b).abs().max()) <= 1e-4 * float(b.abs().max()) + 1e-12
                elif dealt_alike:
                    assert torch.equal(a, b), (wanted, i, k)
                else:
                    # The same products (exact in fp32) summed in another order. A sum is a chain of about 100 additions (a
                    # workgroup's tiles, then the workgroups): rounding errors of sqrt(100) 2^-24 = 6e-7 of partial sums that
                    # are no larger than the largest result (terms of either sign); 16 times that.
                    assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max()), (wanted, i, k)
