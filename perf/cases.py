"""The work that users of this package have it do, as cases that can be timed and compared.

A case is a dict of plain values; its "kind" says which public entry points a pass goes through:

  render      SplatContext.forward in eval mode into buffers that are kept: a serving loop's frame without the net
  frame       a viewer's frame: BlendPointCloud in eval mode, then the reconstruction net, without a graph
  splat_step  SplatContext.forward and .backward into kept buffers, then MyAdamPoints: an optimiser of the splat alone
  train_step  the whole training step through the operator surface: BlendPointCloud with dropout, net, loss, backward,
              MyAdamPoints over the point parameters, MyAdam over net, poses and intrinsics, the pose update
  net_step    the reconstruction net on its own, forward and backward
  adam        MyAdam over the point tensors with one state array per tensor, as the reference keeps it

Clouds have the distributions of trips_amd/scenes.py (uniform cube, normal ball, noisy ground plane with a box above,
tight clusters), made on the GPU. "order" is the memory order of the points: "random", or "morton" for the order that
the reference's scene preprocessing leaves a cloud in (Morton curve, blocks of 256 points shuffled).
"""
import math

import numpy as np
import torch

from trips_amd import abi, scenes
from trips_amd.adam import MyAdam, MyAdamPoints
from trips_amd.renderer import (BlendPointCloud, NeuralRenderInfo, NeuralScene, PointRendererCache, ReducedImageInfo,
                                RenderParams, SplatContext, get_context)
from trips_amd.unet import MultiScaleUnet2dDecOnlySmallFixed, MultiScaleUnet2dParams

BENCH_NET = "16,32,64,64"      # the benchmark's net: four levels
DEFAULT_NET = "32,32,32,32,32"  # MultiScaleUnet2dParams' own: five levels of 32
# Small, so that thousands of passes leave a cloud where it was (the work of a step does not depend on it); smaller where
# the gradients carry the net's fp16 rounding, which through the cameras would soon decide the order of lists.
LR = dict(splat_step=1e-5, train_step=1e-7, adam=1e-3)
LR_CAMERAS = 1e-10


def _case(kind, *, points=0, cloud="plane", order="random", w=0, h=0, layers=8, depth=16, channels=4, views=1, net="",
          steps_bits=32):
    return dict(kind=kind, points=points, cloud=cloud, order=order, w=w, h=h, layers=layers, depth=depth,
                channels=channels, views=views, net=net, steps_bits=steps_bits)


def listed():
    return [
        # the smallest call: a preview frame of a small object, all launches and host time
        dict(name="frame_20k_160x120", **_case("frame", points=20_000, cloud="cube", w=160, h=120, layers=5, net=BENCH_NET)),
        # an object of 100k points at 512 x 512 in a serving loop, short lists
        dict(name="render_100k_512", **_case("render", points=100_000, cloud="cube", w=512, h=512, layers=4, depth=8)),
        # an object of 1M points at full HD
        dict(name="render_1M_1080p", **_case("render", points=1_000_000, cloud="ball", order="morton", w=1920, h=1080)),
        # a viewer's frame of a whole scene at full HD
        dict(name="frame_6M_1080p", **_case("frame", points=6_000_000, order="morton", w=1920, h=1080, net=BENCH_NET)),
        # the splat with 8 descriptor channels on a ragged image, short lists
        dict(name="splat_step_300k_641x479_c8", **_case("splat_step", points=300_000, cloud="ball", w=641, h=479, layers=6,
                                                        depth=8, channels=8)),
        # the splat's benchmark: 6M points in no order, full HD, eight layers
        dict(name="splat_step_6M_1080p", **_case("splat_step", points=6_000_000, w=1920, h=1080)),
        # crowded lists: four views of tight clusters
        dict(name="splat_step_4M_clusters_4views", **_case("splat_step", points=4_000_000, cloud="clusters", w=1245, h=825,
                                                           views=4)),
        # the first steps of a training run on a thinned-out cloud with one small view
        dict(name="train_step_20k_160x120", **_case("train_step", points=20_000, cloud="cube", w=160, h=120, net=BENCH_NET)),
        # the default training load: 512 x 512 crops, four to a step, five layers, the net of five levels
        dict(name="train_step_2M_4crops", **_case("train_step", points=2_000_000, order="morton", w=512, h=512, layers=5,
                                                  views=4, net=DEFAULT_NET)),
        # a training step on whole full-HD images; more points than the packed form of a tile's entries can number
        dict(name="train_step_9M_1080p", **_case("train_step", points=9_000_000, order="morton", w=1920, h=1080,
                                                 net=BENCH_NET)),
        # the net alone on a ragged image, as when the point cloud is frozen
        dict(name="net_step_1245x825", **_case("net_step", w=1245, h=825, layers=5, net=DEFAULT_NET)),
        # the optimiser with the reference's state layout
        dict(name="adam_1M_int64", **_case("adam", points=1_000_000, steps_bits=64)),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("frame", "render", "render", "splat_step", "splat_step", "train_step", "train_step", "net_step", "adam"))
    channels = rng.choice((4, 4, 4, 3, 6, 8, 16))
    points = _log_int(rng, 10_000, 24_000_000 // max(channels, 4))
    if kind == "adam":
        return _case(kind, points=points, channels=channels, steps_bits=rng.choice((32, 64)))
    w = _log_int(rng, 96, 1920)
    h = max(64, int(w * rng.uniform(0.45, 0.75)))
    small = w * h < 600_000
    views = rng.choice((1, 1, 2, 4)) if kind in ("splat_step", "train_step", "net_step") and small else 1
    if views > 1:  # several crops or views to a step
        points = max(10_000, points // views)
    layers = rng.randint(4, 8)
    net = ""
    if kind in ("frame", "train_step", "net_step"):
        levels = rng.randint(3, min(5, layers))
        # a block's outputs are its filters less two images (one at the finest level)
        base = rng.choice((16, 32, 48) if channels <= 4 else (32, 48) if channels <= 8 else (48,)) if small else \
            (16 if channels <= 4 else 32 if channels <= 8 else 48)
        net = ",".join(str(min(64, base * (1 + (i + 1) // 2))) for i in range(levels))
        if kind == "net_step":
            return _case(kind, w=w, h=h, layers=levels, channels=channels, views=views, net=net)
    return _case(kind, points=points, cloud=rng.choice(("cube", "ball", "plane", "clusters")),
                 order=rng.choice(("random", "morton")), w=w, h=h, layers=layers,
                 depth=rng.choice((8, 16, 16)) if kind in ("render", "splat_step") else 16, channels=channels, views=views,
                 net=net)


# ---- inputs -------------------------------------------------------------------------------------------------------

def _uniform(g, shape, lo=0.0, hi=1.0):
    return torch.empty(shape, dtype=torch.float32, device="cuda").uniform_(lo, hi, generator=g)


def _normal(g, shape, sigma=1.0):
    return torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, sigma, generator=g)


def _spread(v):
    """21 bits of v to every third bit."""
    for shift, mask in ((32, 0x1F00000000FFFF), (16, 0x1F0000FF0000FF), (8, 0x100F00F00F00F00F), (4, 0x10C30C30C30C30C3),
                        (2, 0x1249249249249249)):
        v = (v | (v << shift)) & mask
    return v


def _morton_blocks(xyz, g, block=256):
    lo, hi = xyz.amin(dim=0), xyz.amax(dim=0)
    q = ((xyz - lo).double() / (hi - lo).double().clamp_min(1e-30) * (2 ** 21 - 1)).long()
    order = torch.argsort(_spread(q[:, 0]) | (_spread(q[:, 1]) << 1) | (_spread(q[:, 2]) << 2), stable=True)
    n = xyz.shape[0]
    blocks = torch.randperm((n + block - 1) // block, generator=g, device="cuda")
    idx = (blocks[:, None] * block + torch.arange(block, device="cuda")[None, :]).reshape(-1)
    return order[idx[idx < n]]


def _cloud(case, g):
    """xyz, radius, the camera poses and the focal length as a share of the image's width."""
    n, cloud = case["points"], case["cloud"]
    radius = (5e-4, 5e-2)
    if cloud == "cube":
        xyz, radius, focal = _uniform(g, (n, 3), -1.0, 1.0), (1e-3, 3e-2), 500.0 / 512
    elif cloud == "ball":
        xyz, focal = _normal(g, (n, 3), 0.5), 1400.0 / 1920
    elif cloud == "clusters":
        centres = _uniform(g, (64, 3), -1.0, 1.0)
        xyz = centres[torch.randint(64, (n,), generator=g, device="cuda")] + _normal(g, (n, 3), 0.01)
        focal = 1000.0 / 1245
    else:  # "plane": 80 % of the points on a noisy ground plane, the others in a box above it ("up" is -y)
        ground = int(round(0.8 * n))
        xyz = torch.stack([_uniform(g, (n,), -10.0, 10.0),
                           torch.cat([_normal(g, (ground,), 0.02), _uniform(g, (n - ground,), -5.0, 0.0)]),
                           _uniform(g, (n,), -10.0, 10.0)], dim=1)
        xyz = xyz[torch.randperm(n, generator=g, device="cuda")]
        focal = 1400.0 / 1920
    if case["order"] == "morton":
        xyz = xyz[_morton_blocks(xyz, g)]
    poses = []
    for _ in range(case["views"]):
        if cloud == "plane":
            # 1.5 above the ground, outside the cloud: where a point of the box sits in front of the pinhole itself, the
            # last bit of the pose decides its gradient, and no two implementations agree
            a = 2.0 * math.pi * torch.rand(1, generator=g, device="cuda").item() if case["views"] > 1 else 0.0
            away = 15.0 if case["views"] > 1 else 10.5
            poses.append(scenes.look_at_pose((away * math.sin(a), -1.5, -away * math.cos(a)), (0.0, 0.0, 0.0)))
        elif cloud == "clusters":
            d = _normal(g, (3,)).cpu().double().numpy()
            poses.append(scenes.look_at_pose(3.0 * d / np.linalg.norm(d), (0.0, 0.0, 0.0)))
        else:
            poses.append(scenes.look_at_pose((0.3 * len(poses), 0.1 * len(poses), -3.0), (0.0, 0.0, 0.0)))
    r = torch.exp(_uniform(g, (n,), math.log(radius[0]), math.log(radius[1])))
    return xyz, r, np.stack(poses), focal


def _scene(case, g):
    """The tensors of a scene under the operator's names, and its views."""
    xyz, radius, poses, focal = _cloud(case, g)
    n, c, w, h = case["points"], case["channels"], case["w"], case["h"]
    intrinsics = torch.zeros((1, 13), device="cuda")
    intrinsics[0, :4] = torch.tensor([focal * w, focal * w, w / 2.0, h / 2.0])
    t = dict(position=torch.cat([xyz, radius[:, None]], dim=1).contiguous(),
             point_size=torch.log(torch.expm1(radius.double())).float().contiguous(),  # the inverse of the softplus
             index=torch.arange(n, dtype=torch.int32, device="cuda"), texture=_uniform(g, (c, n)),
             confidence=_uniform(g, (n,), 1e-6, 1.0 - 1e-6), background=torch.full((c,), 0.25, device="cuda"),
             poses_se3=torch.as_tensor(poses, dtype=torch.float64, device="cuda").contiguous(), intrinsics=intrinsics)
    views = [dict(w=w, h=h, image_index=i, camera_index=0) for i in range(case["views"])]
    return t, views


def _sizes(case):
    return abi.layer_sizes(case["w"], case["h"], case["layers"])


def _filters(case):
    return [int(f) for f in case["net"].split(",")]


def _net(case, seed):
    f = _filters(case)
    p = MultiScaleUnet2dParams(num_input_layers=case["layers"], num_layers=len(f), num_input_channels=case["channels"],
                               filters_network=f)
    return MultiScaleUnet2dDecOnlySmallFixed(p).he_normal_(torch.Generator().manual_seed(seed)).to("cuda")


def _operator_scene(case, g):
    t, views = _scene(case, g)
    ns = NeuralScene(texture=t["texture"], background_color=t["background"], confidence=t["confidence"].reshape(1, -1),
                     position=t["position"], point_size=t["point_size"].reshape(-1, 1), index=t["index"].reshape(-1, 1),
                     poses_se3=t["poses_se3"], intrinsics=t["intrinsics"])
    info = NeuralRenderInfo(scene=ns, images=[ReducedImageInfo(**v) for v in views],
                            params=RenderParams(max_pixels_per_list=case["depth"], num_texture_channels=case["channels"]),
                            num_layers=case["layers"], train=case["kind"] == "train_step", cache=PointRendererCache())
    return ns, info


def _prepare_frame(case, g, seed):
    ns, info = _operator_scene(case, g)
    net = _net(case, seed)
    net.reuse_packed_weights = True  # a viewer's weights do not change between frames
    return dict(info=info, net=net, scene=ns)


def _prepare_splat(case, g, seed):
    ctx = get_context(0)
    t, views = _scene(case, g)
    train = case["kind"] == "splat_step"
    n, c = case["points"], case["channels"]
    desc = abi.make_desc(num_points=n, num_texels=n, num_channels=c, num_layers=case["layers"], list_depth=case["depth"],
                         views=views, num_images=len(views), num_cameras=1, train=train)
    s = dict(ctx=ctx, desc=desc, t=t, tin=SplatContext.make_in(**t), workspace=ctx.alloc_bytes(ctx.workspace_size(desc)),
             images=ctx.alloc_images(desc), saved=None)
    if train:
        s["saved"] = ctx.alloc_bytes(ctx.saved_size(desc))
        s["grad_images"] = [_normal(g, tuple(im.shape)) for im in s["images"]]
        s["grads"] = dict(d_texture=torch.empty((c, n), device="cuda"), d_confidence=torch.empty(n, device="cuda"),
                          d_background=torch.empty(c, device="cuda"), d_position=torch.empty((n, 4), device="cuda"),
                          d_point_size=torch.empty(n, device="cuda"),
                          d_pose=torch.empty((len(views), 6), dtype=torch.float64, device="cuda"),
                          d_intrinsics=torch.empty((1, 13), device="cuda"))
        s["params"] = [torch.nn.Parameter(t[k]) for k in ("position", "point_size", "texture", "confidence")]
        for p, k in zip(s["params"], ("d_position", "d_point_size", "d_texture", "d_confidence")):
            p.grad = s["grads"][k]
        s["opt"] = MyAdamPoints(s["params"], *s["params"], lr=LR[case["kind"]])
    return s


def _prepare_train(case, g, seed):
    torch.cuda.manual_seed(seed)  # the dropout of a step comes from the default generator
    ns, info = _operator_scene(case, g)
    points = [ns.point_cloud_cuda.t_position, ns.point_cloud_cuda.t_point_size, ns.texture.texture,
              ns.texture.confidence_value_of_point]
    others = [ns.texture.background_color, ns.poses.tangent_poses, ns.intrinsics.intrinsics]
    for p in points + others:
        p.requires_grad_(True)
    net = _net(case, seed)
    net_params = list(net.parameters()) + others
    return dict(ctx=get_context(0), info=info, scene=ns, net=net, points=points, net_params=net_params,
                opt=MyAdamPoints(points, *points, lr=LR["train_step"]),
                net_opt=MyAdam([dict(params=list(net.parameters())), dict(params=others, lr=LR_CAMERAS)], lr=LR["train_step"]),
                target=_uniform(g, (case["views"], 3, case["h"], case["w"])))


def _prepare_net(case, g, seed):
    ins = [_uniform(g, (case["views"], case["channels"], h, w)).requires_grad_(True) for (w, h) in _sizes(case)]
    shape = (case["views"], 3, case["h"], case["w"])
    return dict(net=_net(case, seed), ins=ins, d_out=_normal(g, shape, 1.0 / math.prod(shape)))  # of a mean over the pixels


def _prepare_adam(case, g, seed):
    n, c = case["points"], case["channels"]
    seen = (_uniform(g, (n,)) < 0.61).float()  # the points that a view of the ground plane does not cull
    params = [torch.nn.Parameter(p) for p in (_normal(g, (n, 4)), _normal(g, (n, 1)), _uniform(g, (c, n)), _uniform(g, (1, n)))]
    for p in params:
        p.grad = _normal(g, tuple(p.shape)) * (seen[:, None] if p.shape[0] == n else seen)
    return dict(params=params, opt=MyAdam(params, lr=LR[case["kind"]],
                                          param_steps_dtype=torch.int64 if case["steps_bits"] == 64 else torch.int32))


_PREPARE = dict(frame=_prepare_frame, render=_prepare_splat, splat_step=_prepare_splat, train_step=_prepare_train,
                net_step=_prepare_net, adam=_prepare_adam)


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    state = _PREPARE[case["kind"]](case, g, seed)
    state["kind"] = case["kind"]
    return state


# ---- passes -------------------------------------------------------------------------------------------------------

def _run_frame(s):
    with torch.no_grad():
        images = BlendPointCloud(s["info"])
        return dict(rgb=s["net"].forward(images), images=images)


def _run_render(s):
    s["ctx"].forward(s["desc"], s["tin"], s["images"], None, s["workspace"])
    return s["images"]


def _run_splat_step(s):
    s["ctx"].forward(s["desc"], s["tin"], s["images"], s["saved"], s["workspace"])
    s["ctx"].backward(s["desc"], s["tin"], s["saved"], s["grad_images"], s["grads"], s["workspace"],
                      overwrite_point_grads=True, clear_block_sums=True)
    s["opt"].step()
    return dict(images=s["images"], grads=s["grads"], params=s["params"])


def _run_train_step(s):
    s["opt"].zero_grad(set_to_none=True)
    s["net_opt"].zero_grad(set_to_none=True)
    rgb = s["net"].forward(BlendPointCloud(s["info"]))
    # the squared error: the absolute one's gradient jumps where the image meets its target, so that two correct
    # implementations could not be held against each other
    loss = torch.nn.functional.mse_loss(rgb, s["target"])
    loss.backward()
    s["opt"].step()
    s["net_opt"].step()
    s["ctx"].apply_tangent(s["scene"].poses.tangent_poses.detach(), s["scene"].poses.poses_se3)
    return dict(rgb=rgb, loss=loss, points=s["points"], point_grads=[p.grad for p in s["points"]],
                net_grads=[p.grad for p in s["net_params"]], poses=s["scene"].poses.poses_se3,
                net=torch.nn.utils.parameters_to_vector([p.detach().float() for p in s["net_params"]]))


def _run_net_step(s):
    s["net"].zero_grad(set_to_none=True)
    for t in s["ins"]:
        t.grad = None
    rgb = s["net"].forward(s["ins"])
    rgb.backward(s["d_out"])
    return dict(rgb=rgb, d_ins=[t.grad for t in s["ins"]], d_params=[p.grad for p in s["net"].parameters()])


def _run_adam(s):
    s["opt"].step()
    state = [s["opt"].state[p] for p in s["params"]]
    return dict(params=s["params"], m=[st["first_moments"] for st in state], v=[st["second_moments"] for st in state],
                steps=[st["param_steps"] for st in state])


_RUN = dict(frame=_run_frame, render=_run_render, splat_step=_run_splat_step, train_step=_run_train_step,
            net_step=_run_net_step, adam=_run_adam)


def run(state):
    return _RUN[state["kind"]](state)


# ---- what a pass cannot do without, and how far results may be apart ------------------------------------------------

def _net_flops(case):
    """Of one forward: the 3x3 feature and mask convolutions of every level and the 1x1 at the end."""
    f, c, flops = _filters(case), case["channels"], 0
    for i, (w, h) in enumerate(_sizes(case)[:len(f)]):
        last = i == len(f) - 1
        cin = c if last else c + f[i + 1]
        cout = f[i] - (c if i == 0 else 2 * c)
        flops += 2 * 9 * cin * 2 * cout * w * h
    return case["views"] * (flops + 2 * f[0] * 3 * case["w"] * case["h"])


def work(case):
    kind, n, c, b = case["kind"], case["points"], case["channels"], case["views"]
    elements = n * (6 + c)
    if kind == "adam":
        # weight, gradient, two moments and the counter read, all but the gradient written; 61 % have a gradient
        return dict(bytes=elements * (4 + 0.61 * (24 + 2 * case["steps_bits"] / 8)), flops=elements * 20)
    pixels = b * sum(w * h for (w, h) in _sizes(case))
    pyramid = 4 * c * pixels
    inputs = n * (16 + 4 + 4 + 4 + 4 * c)
    rgb = 12 * b * case["w"] * case["h"]
    if kind == "net_step":
        return dict(bytes=2 * pyramid + 2 * rgb, flops=3 * _net_flops(case))
    if kind == "render":
        return dict(bytes=inputs + pyramid, flops=100 * n * b)
    if kind == "frame":
        return dict(bytes=inputs + pyramid + rgb, flops=100 * n * b + _net_flops(case))
    # a gradient written per parameter; the optimiser reads and writes weights, moments and 32-bit counters
    step = inputs + pyramid + 4 * elements + 28 * elements
    if kind == "splat_step":
        return dict(bytes=step + pyramid, flops=400 * n * b)
    return dict(bytes=step + 2 * rgb, flops=400 * n * b + 3 * _net_flops(case))


def tolerance(case):
    if case["kind"] in ("frame", "train_step", "net_step"):
        # fp16 operands: images and gradients of the net are up to 9e-4 (largest: 5e-3) from its fp32 restatement; the
        # gradients of single points follow the few pixels that they are seen in
        return {"rel": 4e-3, "max": 2e-2 if case["kind"] != "train_step" else 0.4}
    if case["kind"] == "adam":
        return {"rel": 1e-6, "max": 1e-5}
    # 32-bit sums: gradients are up to 4e-6 (largest: 6e-6) from those of the sums in the order of the CPU oracle
    return {"rel": 1.6e-5, "max": 3e-5}
