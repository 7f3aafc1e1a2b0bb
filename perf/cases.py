"""What is timed of this framework: training and mapping passes as user programs run them.

A case is one SOM, one image shape and one call pattern:

  mode     "train": images in order, each seeing the weights the one before it left, then the weights back on the host
           (the reference's loop over Trainer::operator() and update_som()); "map": heatmap and best rotations of every image
  entry    "call":   pink.Trainer / pink.Mapper called once per pink.Data, as a notebook or script loops over its images
           "host":   pink.Trainer.train / pink.Mapper.map on one numpy array
           "device": capi.Context on images that are on the GPU already, results left there
  type     distance type: "float", "uint16", "uint8" (0, 1, 2)
  layout   "cartesian" (som_w x som_h neurons) or "hexagonal" (som_w = som_h = the odd edge)
  channels, image, neuron, region, circular, rotations, flip: the shape of the data and of the distance region
  images   images of one pass

Images are one to four elliptical blobs over a little noise in [0, 1], as cut-outs of surveys look.  A mapper's SOM holds
smooth prototypes that resemble their neighbours, as training leaves them; a trainer starts from uniform noise
(the command line's `--init random`) and goes on from pass to pass.
"""
import math

import numpy as np
import torch

from pink_amd import capi, pink

TYPES = {"float": capi.FLOAT, "uint16": capi.UINT16, "uint8": capi.UINT8}


def _case(name, mode, entry, type, images, layout="cartesian", som_w=10, som_h=10, channels=1, image=64, neuron=44,
          region=32, circular=False, rotations=360, flip=True):
    c = dict(mode=mode, entry=entry, type=type, layout=layout, som_w=som_w, som_h=som_h, channels=channels, image=image,
             neuron=neuron, region=region, circular=circular, rotations=rotations, flip=flip, images=images)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one image through pink.Mapper, the answer awaited: interactive look-ups, a service
        _case("map-call-u8-64px", "map", "call", "uint8", 1),
        # the notebook loop over Trainer::operator() on small images with uint8 pixels and the eight symmetries only
        _case("train-call-u8-28px", "train", "call", "uint8", 250, som_w=8, som_h=8, image=28, neuron=28, region=28, rotations=4),
        # the same SOM trained on one array, as fileio.train_file does a block at a time
        _case("train-host-u8-28px", "train", "host", "uint8", 4000, som_w=8, som_h=8, image=28, neuron=28, region=28, rotations=4),
        # the configuration the headline metric is quoted on
        _case("train-f32-64px", "train", "device", "float", 500),
        # the command line's defaults for 64-pixel images: neuron = image * sqrt(2), region = image * sqrt(2) / 2
        _case("train-host-u8-64px-default", "train", "host", "uint8", 500, neuron=91, region=45),
        # hexagonal SOM, circular region, 16-bit distances
        _case("train-u16-150px-hex", "train", "device", "uint16", 200, layout="hexagonal", som_w=21, som_h=21, image=150,
              neuron=106, region=75, circular=True),
        # three channels, a large SOM, exact float distances
        _case("train-f32-100px-3ch", "train", "device", "float", 100, som_w=40, som_h=40, channels=3, image=100, neuron=70,
              region=50, rotations=180),
        # a survey mapped onto a trained SOM: many images per call
        _case("map-u8-64px", "map", "device", "uint8", 16000),
        _case("map-f32-64px", "map", "device", "float", 1500),
        # an odd number of images, 16-bit distances, hexagonal SOM
        _case("map-u16-150px-hex", "map", "device", "uint16", 301, layout="hexagonal", som_w=21, som_h=21, image=150,
              neuron=106, region=75, circular=True),
        # Radio Galaxy Zoo sized images (124 pixels, hexagonal 21) from host memory
        _case("map-host-u8-124px-hex", "map", "host", "uint8", 1001, layout="hexagonal", som_w=21, som_h=21, image=124,
              neuron=91, region=64),
        # the largest images, the command line's default sizes
        _case("train-u8-256px-default", "train", "device", "uint8", 60, neuron=362, region=181),
    ]


# Limits of a drawn case: what the largest listed cases reach.
_MAX_OPS = 1.1e12            # distance operations of a pass
_MAX_SOM = 24e6              # floats of a SOM
_MAX_IMAGE_FLOATS = 66e6     # floats of a pass's images


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        mode = rng.choice(("train", "map"))
        entry = rng.choice(("device", "device", "device", "host", "host", "call"))
        type = rng.choice(("uint8", "uint16", "float"))
        image = _log(rng, 20, 256)
        # neurons as large as the rotated image, as the image, or as the part every rotation fills
        neuron = max(4, int(round(image * rng.choice((math.sqrt(2), 1.0, math.sqrt(0.5))))))
        region = max(3, min(neuron, int(round(neuron * rng.choice((0.5, math.sqrt(0.5), rng.uniform(0.4, 1.0)))))))
        if rng.random() < 0.25:
            layout, w = "hexagonal", 2 * _log(rng, 2, 10) + 1
            h = w
        else:
            layout, w, h = "cartesian", _log(rng, 3, 40), _log(rng, 3, 40)
        c = _case(None, mode, entry, type, 1, layout, w, h, rng.choice((1, 1, 1, 2, 3)), image, neuron, region,
                  rng.random() < 0.3, rng.choice((4, 360, 360, 180, 4 * _log(rng, 1, 90))), rng.random() < 0.8)
        per_image = _ops(c)
        if _neurons(c) * c["channels"] * neuron ** 2 > _MAX_SOM or per_image > _MAX_OPS / 4 or c["channels"] * region ** 2 > 65000:
            continue
        most = min(_MAX_OPS / per_image, _MAX_IMAGE_FLOATS / (c["channels"] * image ** 2), 16000 if mode == "map" else 4000)
        if entry == "call":
            most = min(most, 250 if mode == "train" else 16)
        c["images"] = max(1, min(int(most), _log(rng, 1, most)))
        return c


def _neurons(c):
    dims = [c["som_w"]] if c["layout"] == "hexagonal" else [c["som_h"], c["som_w"]]
    return capi.som_size(_layout(c), dims)


def _layout(c):
    return capi.HEXAGONAL if c["layout"] == "hexagonal" else capi.CARTESIAN


def _variants(c):
    return c["rotations"] * (2 if c["flip"] else 1)


def _region_elements(c):
    return c["channels"] * c["region"] ** 2 * (math.pi / 4 if c["circular"] else 1.0)


def _ops(c):
    """Distance operations of one image: a subtract-square-accumulate is two."""
    return 2.0 * _neurons(c) * _variants(c) * _region_elements(c)


def work(case):
    """Images read once, results written once, a trainer's SOM read and written once; every (neuron, variant) pair of every
    image evaluated over the region, every base rotation interpolated (11 operations a pixel), the update 3 a weight."""
    c, n = case, case["images"]
    neurons, size = _neurons(c), c["channels"] * c["neuron"] ** 2
    images = 4.0 * n * c["channels"] * c["image"] ** 2
    rotated = 11.0 * n * max(1, c["rotations"] // 4) * size
    if c["mode"] == "map":
        return {"bytes": images + 8.0 * n * neurons + 4.0 * neurons * size, "flops": n * _ops(c) + rotated}
    return {"bytes": images + 8.0 * neurons * size + 4.0 * n, "flops": n * (_ops(c) + 3.0 * neurons * size) + rotated}


def tolerance(case):
    """Integer distances are exact sums and the weight update is a fixed sequence of float32 operations: those results are
    the same bits everywhere.  Float32 distances are 32-bit sums; two candidates that close may change places."""
    if case["type"] == "float":
        return {"rel": 1e-5, "differ": 0.001}
    return "exact"


def _fields(gen, n, channels, dim):
    """n fields of one to four elliptical Gaussian blobs over a little noise, (n, channels, dim, dim) in [0, 1] on the GPU."""
    out = torch.empty((n, channels, dim, dim), device="cuda")
    axis = torch.arange(dim, device="cuda", dtype=torch.float32)
    x, y = axis[None, None, :], axis[None, :, None]
    step = max(1, int(2 ** 24 // (channels * dim * dim)))
    for first in range(0, n, step):
        m = min(step, n - first) * channels
        f = torch.randn((m, dim, dim), device="cuda", generator=gen) * 0.02
        u = torch.rand((4, 7, m, 1, 1), device="cuda", generator=gen)
        for b in range(4):
            cx, cy = (0.2 + 0.6 * u[b, 0]) * dim, (0.2 + 0.6 * u[b, 1]) * dim
            sa, sb = (2 + 10 * u[b, 2]) * dim / 64, (2 + 10 * u[b, 3]) * dim / 64
            t = math.pi * u[b, 4]
            p, q = (x - cx) * torch.cos(t) + (y - cy) * torch.sin(t), (y - cy) * torch.cos(t) - (x - cx) * torch.sin(t)
            present = 1.0 if b == 0 else (u[b, 5] < 0.5).float()
            f += present * (0.3 + 0.7 * u[b, 6]) * torch.exp(-0.5 * ((p / sa) ** 2 + (q / sb) ** 2))
        out[first:first + step] = f.clamp_(0, 1).view(-1, channels, dim, dim)
    return out


def prepare(case, seed):
    c = case
    neurons, channels, dim = _neurons(c), c["channels"], c["neuron"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    images = _fields(gen, c["images"], channels, c["image"])
    if c["image"] <= 32:
        images = torch.floor(images * 255) / 255          # small pictures come with 8-bit pixels
    dims = [c["som_w"]] if c["layout"] == "hexagonal" else [c["som_h"], c["som_w"]]
    functor, sigma, damping = capi.GAUSSIAN, 1.1, 0.2
    factors = capi.make_update_factors(_layout(c), dims, functor, sigma, damping)
    if c["mode"] == "train":
        som = torch.rand((neurons, channels, dim, dim), device="cuda", generator=gen)
    else:
        near = torch.from_numpy(factors).cuda()
        near /= near.sum(1, keepdim=True)
        som = (near @ _fields(gen, neurons, channels, dim).view(neurons, -1)).view(neurons, channels, dim, dim)
    som = som.cpu().numpy()

    if c["entry"] == "device":
        ctx = capi.Context(neurons, channels, c["image"], dim, c["rotations"], c["flip"], c["region"], int(c["circular"]),
                           TYPES[c["type"]], factors if c["mode"] == "train" else None)
        ctx.set_som(som)
        state = {"case": c, "ctx": ctx, "images": images}
        if c["mode"] == "train":
            state["bmu"] = torch.empty(c["images"], dtype=torch.int32, device="cuda")
            state["som"] = np.empty((neurons, channels * dim * dim), np.float32)
        else:
            state["heat"] = torch.empty((c["images"], neurons), device="cuda")
            state["best"] = torch.empty((c["images"], neurons), dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        return state

    neuron_shape = (dim, dim) if channels == 1 else (channels, dim, dim)
    image_shape = (c["image"],) * 2 if channels == 1 else (channels, c["image"], c["image"])
    layout = "cartesian-2d" if channels == 1 else "cartesian-3d"
    som_shape = (neurons,) if c["layout"] == "hexagonal" else (c["som_h"], c["som_w"])
    som = pink.SOM(som.reshape(som_shape + neuron_shape), som_layout=c["layout"] + "-2d", neuron_layout=layout)
    options = dict(number_of_rotations=c["rotations"], use_flip=c["flip"], euclidean_distance_dim=c["region"],
                   euclidean_distance_shape=pink.EuclideanDistanceShape(int(c["circular"])),
                   euclidean_distance_type=pink.DataType(TYPES[c["type"]]))
    if c["mode"] == "train":
        tool = pink.Trainer(som, pink.GaussianFunctor(sigma, damping), **options)
    else:
        tool = pink.Mapper(som, **options)
    return {"case": c, "som": som, "tool": tool, "layout": layout, "images": images.cpu().numpy().reshape((-1,) + image_shape)}


def run(state):
    c = state["case"]
    train = c["mode"] == "train"
    if c["entry"] == "device":
        ctx = state["ctx"]
        if train:
            ctx.train_device(state["images"].data_ptr(), c["images"], state["bmu"].data_ptr())
            ctx.get_som(state["som"])                      # waits for the training
            return {"bmu": state["bmu"], "som": state["som"]}
        ctx.map_device(state["images"].data_ptr(), c["images"], state["heat"].data_ptr(), state["best"].data_ptr())
        ctx.synchronize()                                  # the results are complete for whatever stream reads them next
        return {"heatmap": state["heat"], "best": state["best"]}

    tool, images, layout = state["tool"], state["images"], state["layout"]
    if c["entry"] == "host":
        if not train:
            heatmap, best = tool.map(images, layout)
            return {"heatmap": heatmap, "best": best}
        bmu = tool.train(images, layout)
        tool.update_som()
        return {"bmu": bmu, "som": np.asarray(state["som"])}
    if not train:
        answers = [tool(pink.Data(image, layout=layout)) for image in images]
        return {"heatmap": np.array([a[0] for a in answers], np.float32), "best": np.array([a[1] for a in answers], np.uint32)}
    for image in images:
        tool(pink.Data(image, layout=layout))
    tool.update_som()
    return {"counts": tool.update_info, "som": np.asarray(state["som"])}
