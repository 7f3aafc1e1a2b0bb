"""GPU parity: the HIP path through the C ABI against the CPU oracle.

Bars (stated where checked): rotated pixels bit-exact; float32 distances bit-exact
with the oracle (stricter than the 1e-5 relative gate) and best rotation / BMU
identical; integer sums, best rotations and BMUs bit-exact; trained weights
bit-exact after several sequential images (gate: 1e-4 absolute).
"""
import sys

import numpy as np
import pytest

import oracle as O
from pink_amd import capi, synthetic

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


ROT_SHAPES = [
    # C, I, D, num_rot, flip
    (1, 64, 44, 360, True), (1, 150, 106, 360, True), (3, 100, 70, 180, True), (1, 28, 28, 4, True),
    (1, 64, 45, 360, True), (1, 64, 100, 360, True), (1, 124, 91, 360, True), (2, 17, 24, 16, False),
    (1, 2, 4, 1, False), (1, 4, 2, 8, True), (1, 5, 3, 360, False), (3, 9, 9, 1, True),
    (1, 200, 141, 8, True),     # a base rotation of 78 KiB in LDS
    (1, 290, 205, 8, True),     # 205*205*4 B > 158 KiB and so is the image: nothing in LDS
    (1, 150, 205, 16, True),    # the image in LDS instead of the base rotation
    (2, 160, 226, 8, False),
    (1, 210, 260, 8, True),     # nothing in LDS, neurons larger than the image
]


@pytest.mark.parametrize("C_,I,D,nrot,flip", ROT_SHAPES)
def test_rotate_bit_exact(C_, I, D, nrot, flip):
    say("rotate", C_, I, D, nrot, flip)
    rng = np.random.default_rng(I * 1000 + D + nrot)
    img = rng.random((C_, I, I), dtype=np.float32)
    with capi.Context(3, C_, I, D, nrot, flip, min(D, 2)) as ctx:
        got = ctx.rotate(img)
    want = O.rotated_images(img, C_, I, D, nrot, flip)
    assert np.array_equal(bits(got), bits(want))


@pytest.mark.parametrize("ed_type", [capi.UINT8, capi.UINT16])
def test_rotate_tap_on_integer_contexts_with_channels(ed_type):
    # integer contexts keep the base rotations of all channels in one block of the rotation kernel
    C_, I, D, nrot, flip = 3, 20, 14, 8, True
    say("rotate tap, integer, channels", ed_type)
    rng = np.random.default_rng(ed_type)
    img = rng.random((C_, I, I), dtype=np.float32)
    want = O.rotated_images(img, C_, I, D, nrot, flip)
    F = capi.make_update_factors(capi.CARTESIAN, [3], capi.GAUSSIAN, 1.0, 0.5)
    for factors in (None, F):
        with capi.Context(3, C_, I, D, nrot, flip, 9, capi.QUADRATIC, ed_type, factors) as ctx:
            assert np.array_equal(bits(ctx.rotate(img)), bits(want))


def test_rotate_reference_golden():
    # test/SelfOrganizingMapTest/generate_rotated_images.cpp:15-41
    with capi.Context(1, 1, 2, 2, 4, False, 2) as ctx:
        out = ctx.rotate(np.array([1, 2, 3, 4], np.float32))
    assert out.ravel().tolist() == [1, 2, 3, 4, 3, 1, 4, 2, 4, 3, 2, 1, 2, 4, 1, 3]
    with capi.Context(1, 2, 2, 2, 4, False, 2) as ctx:
        out = ctx.rotate(np.arange(1, 9, dtype=np.float32))
    assert out.ravel().tolist() == [1, 2, 3, 4, 5, 6, 7, 8, 3, 1, 4, 2, 7, 5, 8, 6,
                                    4, 3, 2, 1, 8, 7, 6, 5, 2, 4, 1, 3, 6, 8, 5, 7]


DIST_SHAPES = [
    # N, C, I, D, nrot, flip, ed, shape
    (100, 1, 64, 44, 360, True, 32, capi.QUADRATIC),      # cfg 0 / 1
    (64, 1, 28, 28, 4, True, 28, capi.QUADRATIC),         # cfg 4
    (37, 1, 40, 29, 16, True, 21, capi.CIRCULAR),
    (9, 2, 17, 24, 8, False, 13, capi.QUADRATIC),
    (9, 2, 17, 24, 8, True, 13, capi.CIRCULAR),           # 3-D circular: channel 0 counted twice (CPU rule)
    (4, 1, 8, 8, 1, False, 8, capi.QUADRATIC),
    (5, 1, 8, 8, 1, True, 5, capi.QUADRATIC),
    (331, 1, 150, 106, 360, True, 75, capi.CIRCULAR),     # cfg 2
    (1600, 3, 100, 70, 180, True, 50, capi.QUADRATIC),    # cfg 3
    (7, 1, 40, 28, 720, True, 20, capi.QUADRATIC),        # 1440 variants: six row tiles of base rotations
    (3, 1, 30, 20, 1024, False, 15, capi.CIRCULAR),       # eight
    (5, 1, 160, 226, 8, True, 113, capi.QUADRATIC),       # neurons too large for an LDS tile: the image in LDS
    (5, 1, 290, 205, 8, True, 40, capi.CIRCULAR),         # ... nothing in LDS
    (4, 1, 210, 297, 12, True, 148, capi.QUADRATIC),      # ... and neurons larger than the image
    (5, 1, 128, 181, 16, True, 90, capi.QUADRATIC),       # a 128 KiB base rotation in LDS
]


def _som_and_image(N, C_, I, D, seed):
    rng = np.random.default_rng(seed)
    som = rng.random((N, C_ * D * D), dtype=np.float32)
    img = rng.random((C_, I, I), dtype=np.float32)
    return som, img


@pytest.mark.parametrize("ed_type", [capi.FLOAT, capi.UINT8, capi.UINT16])
@pytest.mark.parametrize("N,C_,I,D,nrot,flip,ed,shape_", DIST_SHAPES)
def test_distance_parity(N, C_, I, D, nrot, flip, ed, shape_, ed_type):
    say("distance", N, C_, I, D, nrot, flip, ed, shape_, ed_type)
    som, img = _som_and_image(N, C_, I, D, N + D + ed)
    if N < 331:
        som[1] = O.rotated_images(img, C_, I, D, nrot, flip)[min(3, nrot - 1)].ravel()   # an exact match
        som[2] = som[1] * np.float32(0.5)
    s = O.shape(N, C_, I, D, nrot, flip, ed, shape_, ed_type)
    rot = O.rotated_images(img, C_, I, D, nrot, flip)
    od, ossd, obest = O.distance_matrix(s, som, rot)
    # a uint8 mapper runs on the matrix cores where a kernel applies: check every kernel
    choices = [capi.KERNEL_AUTO]
    if ed_type == capi.UINT8:
        choices += [capi.KERNEL_VALU, capi.KERNEL_MFMA, capi.KERNEL_MFMA_SYM, capi.KERNEL_MFMA_GEMM]
    if ed_type == capi.UINT16:
        choices += [capi.KERNEL_VALU, capi.KERNEL_MFMA_GEMM]
    ran = 0
    for choice in choices:
        try:
            ctx = capi.Context(N, C_, I, D, nrot, flip, ed, shape_, ed_type, kernel_choice=choice)
        except capi.PinkError:
            assert choice in (capi.KERNEL_MFMA, capi.KERNEL_MFMA_SYM)    # refused: shape outside that kernel
            continue
        ran += 1
        with ctx:
            ctx.set_som(som)
            assert ctx.region_size == len(O.region(C_, D, ed, shape_))
            d, ssd, best = ctx.distance(img)
        if ed_type == capi.FLOAT:
            # gate: 1e-5 relative, argmin identical up to ties; achieved and asserted: bit-exact
            assert np.array_equal(bits(d), bits(od))
        else:
            assert np.array_equal(ssd, ossd), choice
            assert np.array_equal(bits(d), bits(od)), choice
        assert np.array_equal(best, obest), choice


# The float32 distance kernel has two forms chosen by the amount of work per launch: neuron values by DPP
# broadcast (blocks of one neuron per wave, while they are all resident at once) and neuron values as scalar
# operands with two or four neurons per wave.  Same chains, same order: every form is bit-equal to the oracle.
@pytest.mark.parametrize("N,C_,I,D,nrot,flip,ed,shape_,n_map", [
    (397, 1, 64, 44, 360, True, 32, capi.QUADRATIC, 0),      # one image: scalar operands, two neurons per wave
    (1597, 1, 64, 44, 360, True, 32, capi.QUADRATIC, 0),     # one image: four neurons per wave
    (70, 1, 20, 14, 32, True, 9, capi.CIRCULAR, 300),        # a launch group of small images: four neurons per wave, two stages
    (37, 1, 40, 29, 16, True, 21, capi.CIRCULAR, 150),       # ... two neurons per wave, neuron count not a multiple of 8
])
def test_float32_distance_forms(N, C_, I, D, nrot, flip, ed, shape_, n_map):
    say("float32 distance forms", N, C_, I, D, nrot, flip, ed, shape_, n_map)
    rng = np.random.default_rng(N * 31 + n_map)
    som = rng.random((N, C_ * D * D), dtype=np.float32)
    s = O.shape(N, C_, I, D, nrot, flip, ed, shape_, capi.FLOAT)
    with capi.Context(N, C_, I, D, nrot, flip, ed, shape_, capi.FLOAT) as ctx:
        ctx.set_som(som)
        if n_map == 0:
            img = rng.random((C_, I, I), dtype=np.float32)
            som[N // 2] = O.rotated_images(img, C_, I, D, nrot, flip)[min(5, nrot - 1)].ravel()   # an exact match
            ctx.set_som(som)
            od, _, obest = O.distance_matrix(s, som, O.rotated_images(img, C_, I, D, nrot, flip))
            d, _, best = ctx.distance(img)
            assert np.array_equal(bits(d), bits(od))
            assert np.array_equal(best, obest)
        else:
            imgs = rng.random((n_map, C_, I, I), dtype=np.float32)
            heat, best = ctx.map(imgs)
            oheat, obest = O.map_images(s, som, imgs)
            assert np.array_equal(bits(heat), bits(oheat))
            assert np.array_equal(best, obest)


TRAIN_CASES = [
    # workload, images, ed_type override, distance kernel
    ("cfg0", 6, None, capi.KERNEL_AUTO), ("cfg4", 40, None, capi.KERNEL_AUTO), ("cfg4", 10, None, capi.KERNEL_VALU),
    ("cfg0", 4, capi.UINT8, capi.KERNEL_AUTO), ("cfg0", 3, capi.UINT8, capi.KERNEL_VALU),
    ("cfg0", 3, capi.UINT16, capi.KERNEL_AUTO), ("cfg2", 3, None, capi.KERNEL_AUTO), ("cfg2", 1, None, capi.KERNEL_VALU),
    ("cfg3", 1, None, capi.KERNEL_AUTO),
]


@pytest.mark.parametrize("name,n,ed_type,choice", TRAIN_CASES)
def test_train_parity(name, n, ed_type, choice):
    w = synthetic.WORKLOADS[name]
    ed_type = w.ed_type if ed_type is None else ed_type
    say("train", name, n, ed_type, choice)
    imgs = synthetic.images(w, n)
    som0 = synthetic.initial_som(w)
    F = synthetic.update_factors(w)
    with capi.Context(w.som_size, w.channels, w.image_dim, w.neuron_dim, w.num_rot, w.use_flip, w.ed_dim,
                      w.ed_shape, ed_type, F, kernel_choice=choice) as ctx:
        ctx.set_som(som0)
        bmu = ctx.train(imgs)
        got = ctx.get_som()
    s = O.shape(w.som_size, w.channels, w.image_dim, w.neuron_dim, w.num_rot, w.use_flip, w.ed_dim,
                w.ed_shape, ed_type)
    want = som0.copy()
    obmu = O.train(s, want, imgs, F)
    assert np.array_equal(bmu, obmu)
    # gate: 1e-4 absolute (test/CudaTest/compare_trainer_cpu.cu:76); asserted: bit-exact
    assert np.abs(got - want).max() <= 1e-4
    assert np.array_equal(bits(got), bits(want))


def test_train_one_call_per_image_equals_batched_call():
    w = synthetic.WORKLOADS["cfg4"]
    imgs = synthetic.images(w, 12)
    som0 = synthetic.initial_som(w)
    with synthetic.make_context(w) as a, synthetic.make_context(w) as b:
        a.set_som(som0)
        b.set_som(som0)
        bm_a = a.train(imgs)
        bm_b = np.concatenate([b.train(imgs[i]) for i in range(len(imgs))])
        assert np.array_equal(bm_a, bm_b)
        assert np.array_equal(bits(a.get_som()), bits(b.get_som()))


@pytest.mark.parametrize("name,n", [("cfg0", 150), ("cfg4", 200)])
def test_calls_without_a_result_train_in_order_whatever_comes_between(name, n):
    """Calls that hand nothing back (the reference's Trainer::operator()) are collected into launch groups;
    every other call on the context first trains what is pending.  Weights, best matches and counts are those of
    one call over all images, and of the CPU."""
    w = synthetic.WORKLOADS[name]
    imgs = synthetic.images(w, n)
    som0 = synthetic.initial_som(w)
    F = synthetic.update_factors(w)
    s = O.shape(w.som_size, w.channels, w.image_dim, w.neuron_dim, w.num_rot, w.use_flip, w.ed_dim, w.ed_shape, w.ed_type)
    with synthetic.make_context(w) as ctx:
        ctx.set_som(som0)
        bmu_mid = None
        for i in range(n):
            if i == 70:
                d_mid = ctx.distance(imgs[0])[0]          # sees the SOM after 70 images
            if i == 100:
                bmu_mid = ctx.train(imgs[100:103])         # a call with a result, in the middle of pending ones
                continue
            if i in (101, 102):
                continue
            if i == 120:
                ctx.rotate(imgs[5])                        # the debug tap shares buffers with the trainer
            ctx.train(imgs[i], want_bmu=False)             # three of them in one call further down
        counts = ctx.update_counts()
        got = ctx.get_som()
    want = som0.copy()
    obmu = O.train(s, want, imgs, F)
    assert np.array_equal(bits(got), bits(want))
    assert np.array_equal(bmu_mid, obmu[100:103])
    assert np.array_equal(counts, np.bincount(obmu, minlength=w.som_size))
    mid = som0.copy()
    O.train(s, mid, imgs[:70], F)
    od = O.distance_matrix(s, mid, O.rotated_images(imgs[0], w.channels, w.image_dim, w.neuron_dim, w.num_rot, w.use_flip))[0]
    assert np.array_equal(bits(d_mid), bits(od))


@pytest.mark.parametrize("name", ["cfg4", "cfg0"])
def test_rotation_tap_between_training_calls(name):
    # a trainer keeps two of a base rotation's eight symmetries; the tap asks for all of them in between
    w = synthetic.WORKLOADS[name]
    say("tap between training calls", name)
    imgs = synthetic.images(w, 6)
    som0 = synthetic.initial_som(w)
    with synthetic.make_context(w) as a, synthetic.make_context(w) as b:
        a.set_som(som0)
        b.set_som(som0)
        bm_a = a.train(imgs)
        first = b.train(imgs[:3])
        variants = b.rotate(imgs[5])
        second = b.train(imgs[3:])
        want = O.rotated_images(imgs[5], w.channels, w.image_dim, w.neuron_dim, w.num_rot, w.use_flip)
        assert np.array_equal(bits(variants), bits(want))
        assert np.array_equal(bm_a, np.concatenate([first, second]))
        assert np.array_equal(bits(a.get_som()), bits(b.get_som()))


def test_reference_trainer_known_answers():
    # test/SelfOrganizingMapTest/Trainer.cpp:49-94 and test/CudaTest/update_neurons.cu:16-41
    F = capi.make_update_factors(capi.CARTESIAN, [2, 2], capi.GAUSSIAN, 1.1, 0.2, 0.0)
    with capi.Context(4, 1, 2, 2, 1, False, 2, update_factors=F) as ctx:
        ctx.set_som(np.zeros((4, 4), np.float32))
        ctx.train(np.array([1000, 2000, 3000, 4000], np.float32))
        assert int(ctx.get_som()[0, 3]) == 290
    F = capi.make_update_factors(capi.CARTESIAN, [1, 1], capi.STEP, 10.0)
    with capi.Context(1, 1, 4, 2, 1, False, 2, update_factors=F) as ctx:
        ctx.set_som(np.zeros((1, 4), np.float32))
        ctx.train(np.arange(1, 17, dtype=np.float32))
        assert ctx.get_som().ravel().tolist() == [6, 7, 10, 11]
    F = capi.make_update_factors(capi.CARTESIAN, [2, 2], capi.STEP, 0.0)
    with capi.Context(4, 2, 2, 2, 4, False, 2, update_factors=F) as ctx:
        som = np.zeros((4, 8), np.float32)
        som[1] = [4, 3, 2, 1, 8, 7, 6, 5]
        ctx.set_som(som)
        bmu = ctx.train(np.arange(1, 9, dtype=np.float32))
        assert bmu.tolist() == [1] and np.array_equal(ctx.get_som(), som)


MAP_CASES = [("cfg1", 24, None, capi.KERNEL_AUTO), ("cfg1", 9, None, capi.KERNEL_VALU),
             ("cfg1", 13, None, capi.KERNEL_MFMA), ("cfg1", 40, None, capi.KERNEL_MFMA_SYM),
             ("cfg0", 5, capi.FLOAT, capi.KERNEL_AUTO),
             ("cfg4", 300, None, capi.KERNEL_AUTO), ("cfg4", 50, None, capi.KERNEL_VALU),
             ("cfg2", 2, None, capi.KERNEL_AUTO)]


@pytest.mark.parametrize("name,n,ed_type,choice", MAP_CASES)
def test_map_parity(name, n, ed_type, choice):
    w = synthetic.WORKLOADS[name]
    ed_type = w.ed_type if ed_type is None else ed_type
    say("map", name, n, ed_type, choice)
    imgs = synthetic.images(w, n)
    som = synthetic.initial_som(w)
    som[3] = O.rotated_images(imgs[1], w.channels, w.image_dim, w.neuron_dim, w.num_rot, w.use_flip)[5 % w.R].ravel()
    with capi.Context(w.som_size, w.channels, w.image_dim, w.neuron_dim, w.num_rot, w.use_flip, w.ed_dim,
                      w.ed_shape, ed_type, None, max_batch=7, kernel_choice=choice) as ctx:
        ctx.set_som(som)
        heat, best = ctx.map(imgs)
    s = O.shape(w.som_size, w.channels, w.image_dim, w.neuron_dim, w.num_rot, w.use_flip, w.ed_dim,
                w.ed_shape, ed_type)
    oheat, obest = O.map_images(s, som, imgs)
    assert np.array_equal(bits(heat), bits(oheat))
    assert np.array_equal(best, obest)


SYM_SHAPES = [
    # N, C, I, D, nrot, flip, ed, shape, images   -- each exercises another corner of the resident-SOM kernels
    (3, 1, 24, 18, 40, True, 16, capi.QUADRATIC, 5),       # 8 k-steps, one unit per image, one column tile, batch not a multiple of 4
    (70, 1, 32, 24, 160, True, 22, capi.QUADRATIC, 9),     # 16 k-steps, two units per image, three SOM slices
    (150, 1, 45, 32, 360, True, 27, capi.QUADRATIC, 3),    # 24 k-steps, three units, five slices, image edge not a multiple of 4
    (33, 1, 40, 44, 360, False, 32, capi.QUADRATIC, 37),   # 32 k-steps, padded neurons (I < D), no flip, more images than one group
    (20, 2, 20, 16, 8, True, 10, capi.QUADRATIC, 6),       # two channels, two base rotations
    (12, 1, 16, 12, 4, True, 12, capi.QUADRATIC, 4),       # quarter turns only
    (12, 1, 16, 12, 1, True, 12, capi.QUADRATIC, 4),       # flip only
    (25, 1, 40, 29, 16, True, 21, capi.CIRCULAR, 7),       # circular region, odd diameter
    (1, 1, 28, 28, 360, True, 28, capi.QUADRATIC, 1),      # a single neuron, a single image
    (3, 2, 6, 7, 360, True, 1, capi.QUADRATIC, 3),         # a one-pixel region: equal distances all over, the first variant wins
    (37, 1, 64, 91, 360, True, 45, capi.QUADRATIC, 9),     # 2025 elements: the wide form (64 k-steps, one column tile per wave)
    (130, 1, 64, 64, 360, True, 44, capi.CIRCULAR, 2),     # wide form, 48 k-steps, nine slices
    (9, 1, 52, 42, 360, True, 38, capi.QUADRATIC, 40),     # wide form, several images per group
    (20, 2, 40, 30, 360, False, 30, capi.QUADRATIC, 4),    # wide form, two channels, no flip
    (40, 1, 24, 18, 40, True, 16, capi.QUADRATIC, 600),    # ten column tiles: a whole block and two tiles for the kernel that splits k, more images than its blocks
    (100, 1, 45, 32, 72, True, 27, capi.QUADRATIC, 5),     # 25 column tiles at 24 k-steps: three blocks and one tile
]


@pytest.mark.parametrize("N,C_,I,D,nrot,flip,ed,shape_,n", SYM_SHAPES)
def test_map_uint8_kernels_over_shapes(N, C_, I, D, nrot, flip, ed, shape_, n):
    say("map u8 shapes", N, C_, I, D, nrot, flip, ed, shape_, n)
    rng = np.random.default_rng(N * 7 + I + nrot)
    som = rng.random((N, C_ * D * D), dtype=np.float32)
    imgs = rng.random((n, C_, I, I), dtype=np.float32)
    R = nrot * (2 if flip else 1)
    som[N // 2] = O.rotated_images(imgs[0], C_, I, D, nrot, flip)[R - 1].ravel()       # an exact match at the last variant
    s = O.shape(N, C_, I, D, nrot, flip, ed, shape_, capi.UINT8)
    oheat, obest = O.map_images(s, som, imgs)
    ran = []
    for choice in (capi.KERNEL_AUTO, capi.KERNEL_MFMA_SYM, capi.KERNEL_MFMA, capi.KERNEL_MFMA_GEMM):
        try:
            ctx = capi.Context(N, C_, I, D, nrot, flip, ed, shape_, capi.UINT8, None, max_batch=16, kernel_choice=choice)
        except capi.PinkError:
            assert choice in (capi.KERNEL_MFMA, capi.KERNEL_MFMA_SYM)
            continue
        with ctx:
            ran.append(ctx.distance_kernel)
            ctx.set_som(som)
            heat, best = ctx.map(imgs)
            heat_again, best_again = ctx.map(imgs[:1])        # a second, shorter call on the same context
        assert np.array_equal(bits(heat), bits(oheat)), choice
        assert np.array_equal(best, obest), choice
        assert np.array_equal(bits(heat_again), bits(oheat[:1])) and np.array_equal(best_again, obest[:1]), choice
    say("   kernels that ran:", ran)
    assert capi.KERNEL_MFMA_GEMM in ran and capi.KERNEL_MFMA_SYM in ran


ORBIT_MAP_SHAPES = [
    # N, C, I, D, num_rot, flip, ed, shape, type, images, data
    (5, 1, 12, 9, 1, True, 7, capi.QUADRATIC, capi.UINT16, 3, "noise"),       # no quarter turns; an odd neuron
    (70, 1, 60, 54, 4, True, 48, capi.QUADRATIC, capi.UINT8, 67, "noise"),    # one row per image: 32 images in a row tile
    (9, 1, 61, 60, 12, False, 51, capi.QUADRATIC, capi.UINT8, 5, "noise"),    # four columns per neuron, unlike symmetries
    (33, 2, 20, 14, 132, True, 10, capi.QUADRATIC, capi.UINT16, 9, "noise"),  # 33 rows per image: tiles of two images
    (17, 1, 40, 57, 360, False, 41, capi.CIRCULAR, capi.UINT16, 4, "noise"),
    (3, 1, 180, 254, 8, True, 181, capi.QUADRATIC, capi.UINT8, 1, "noise"),   # an image beyond the LDS, k in splits
    (90, 1, 16, 12, 360, True, 8, capi.QUADRATIC, capi.UINT16, 300, "noise"), # the large tiles
    (340, 1, 70, 64, 360, True, 60, capi.CIRCULAR, capi.UINT8, 4, "noise"),
    (4, 1, 1, 6, 12, True, 5, capi.QUADRATIC, capi.UINT16, 3, "noise"),       # an image of a pixel
    (6, 2, 61, 40, 68, True, 25, capi.QUADRATIC, capi.UINT16, 5, "noise"),    # a window of the image; pieces partly outside the region
    (5, 1, 250, 64, 40, False, 37, capi.CIRCULAR, capi.UINT8, 4, "noise"),    # ... of an image beyond the LDS
    (9, 1, 24, 18, 128, True, 13, capi.QUADRATIC, capi.FLOAT, 5, "noise"),    # 13 rows and columns: bands and patches cut short
    (6, 3, 20, 15, 360, False, 9, capi.QUADRATIC, capi.FLOAT, 3, "noise"),
    (37, 1, 30, 30, 456, True, 30, capi.CIRCULAR, capi.FLOAT, 6, "noise"),    # 114 rows: more than the kept ones
    (13, 1, 150, 106, 72, True, 75, capi.CIRCULAR, capi.FLOAT, 2, "noise"),
    (40, 1, 20, 14, 360, True, 10, capi.QUADRATIC, capi.FLOAT, 4, "flat"),    # every variant ties
    (40, 1, 20, 14, 360, True, 10, capi.QUADRATIC, capi.FLOAT, 4, "mask"),    # values that rounding keeps, many ties
    (5, 1, 12, 8, 128, True, 5, capi.QUADRATIC, capi.FLOAT, 1500, "thirds"),  # more images than are counted at a time
    (70, 1, 30, 24, 360, False, 17, capi.QUADRATIC, capi.FLOAT, 60, "thirds"),  # two runs of 64 neurons, four columns per neuron
    (40, 1, 20, 14, 360, True, 10, capi.QUADRATIC, capi.FLOAT, 150, "grown"),  # some neurons of an image keep every variant
    (12, 1, 20, 14, 360, True, 10, capi.QUADRATIC, capi.FLOAT, 4, "wide"),    # either sign, six orders of magnitude
    (12, 1, 20, 14, 360, True, 10, capi.QUADRATIC, capi.FLOAT, 4, "tiny"),    # squares below the smallest normal number
]


@pytest.mark.parametrize("N,C_,I,D,nrot,flip,ed,shape_,ed_type,n,data", ORBIT_MAP_SHAPES)
def test_map_with_orbit_rows(N, C_, I, D, nrot, flip, ed, shape_, ed_type, n, data):
    """Mappers whose rows are base rotations in the order of the symmetries' orbits; float32 distances are screened on rounded
    values first, the variants that can be a neuron's closest are then summed exactly.  A call with few float32 images sums every
    variant instead: the images come often enough here that the call screens them, and a single one that is summed."""
    say("orbit mapper", N, C_, I, D, nrot, flip, ed, shape_, ed_type, n, data)
    rng = np.random.default_rng(N * 7 + I + nrot)
    imgs, som = rng.random((n, C_, I, I), dtype=np.float32), rng.random((N, C_ * D * D), dtype=np.float32)
    if data == "flat":
        imgs[:], som[:] = 0.25, 0.5
    elif data == "thirds":
        imgs[::3] = 0.25
    elif data == "grown":
        som[::7] *= 3000.0
    elif data == "mask":
        imgs, som = (imgs < 0.1).astype(np.float32), (som < 0.1).astype(np.float32)
    elif data == "wide":
        imgs, som = ((imgs - 0.5) * 10.0 ** rng.integers(-3, 4, imgs.shape)).astype(np.float32), ((som - 0.5) * 300).astype(np.float32)
    elif data == "tiny":
        imgs, som = imgs * np.float32(1e-33), som * np.float32(1e-21)
    s = O.shape(N, C_, I, D, nrot, flip, ed, shape_, ed_type)
    want_heat, want_best = O.map_images(s, som, imgs)
    with capi.Context(N, C_, I, D, nrot, flip, ed, shape_, ed_type) as ctx:
        ctx.set_som(som)
        times = 1
        if ed_type == capi.FLOAT:
            variant_elements = nrot * (2 if flip else 1) * ctx.region_size
            times += int((9.0 + 0.021 * ctx.region_size) / (1.7e-6 * variant_elements)) // n
        heat, best = ctx.map(np.tile(imgs, (times, 1, 1, 1)))
        one_heat, one_best = ctx.map(imgs[-1:])
    for t in range(times):
        part = slice(t * n, (t + 1) * n)
        assert np.array_equal(best[part], want_best) and np.array_equal(bits(heat[part]), bits(want_heat)), t
    assert np.array_equal(one_best, want_best[-1:]) and np.array_equal(bits(one_heat), bits(want_heat[-1:]))


@pytest.mark.parametrize("N,C_,I,D,nrot,flip,ed,n", [
    (9, 1, 24, 18, 128, True, 13, 400),                                # regions that are not symmetric, shorter than a step of the product
    (6, 3, 20, 15, 360, False, 9, 300),
    (9, 1, 40, 30, 64, True, 16, 300),                                 # 16 base rotations, the fewest that are screened
    (600, 1, 16, 12, 64, True, 10, 120),                               # summed however many images come
    (520, 1, 30, 24, 360, True, 20, 270),                              # more pairs than one wave's blocks of the selection take
])
def test_map_of_many_images(N, C_, I, D, nrot, flip, ed, n):
    """Float32 mappers on either side of the line where screening pays, and of the selection's forms."""
    say("float mapper, many images", N, C_, I, D, nrot, flip, ed, n)
    rng = np.random.default_rng(N + D)
    imgs, som = rng.random((n, C_, I, I), dtype=np.float32), rng.random((N, C_ * D * D), dtype=np.float32)
    few = min(n, 40)
    want_heat, want_best = O.map_images(O.shape(N, C_, I, D, nrot, flip, ed, capi.QUADRATIC, capi.FLOAT), som, imgs[:few])
    with capi.Context(N, C_, I, D, nrot, flip, ed, capi.QUADRATIC, capi.FLOAT) as ctx:
        ctx.set_som(som)
        heat, best = ctx.map(imgs)
        parts = [ctx.map(imgs[i:i + 2]) for i in range(0, n, 2)]
    assert np.array_equal(best[:few], want_best) and np.array_equal(bits(heat[:few]), bits(want_heat))
    assert np.array_equal(best, np.concatenate([p[1] for p in parts])) and np.array_equal(bits(heat), bits(np.concatenate([p[0] for p in parts])))


@pytest.mark.parametrize("N,I,D,nrot,ed,train", [
    (40, 20, 14, 360, 10, False),
    (40, 20, 14, 360, 9, False),                                       # not symmetric
    (9, 100, 96, 360, 91, True),
    (900, 40, 34, 360, 32, True),
])
def test_screening_with_infinities(monkeypatch, N, I, D, nrot, ed, train):
    """Infinite pixels and weights bound nothing; against the kernel that sums every variant."""
    monkeypatch.setenv("PINK_HIP_RESIDENT_TRAINER", "0")
    say("screening with infinities", N, I, D, nrot, ed, train)
    n = 12 if train else 150
    rng = np.random.default_rng(N + ed)
    som, imgs = rng.random((N, D, D), dtype=np.float32), rng.random((n, 1, I, I), dtype=np.float32)
    imgs[3, 0, I // 2, I // 2], imgs[n // 2, 0, I // 2, I // 2 - 2] = np.inf, -np.inf
    som[::5, D // 2, D // 2], som[3::5, D // 2, D // 2 + 1] = np.inf, -np.inf
    F = capi.make_update_factors(capi.CARTESIAN, [N], capi.GAUSSIAN, 1.0, 0.5) if train else None
    got = []
    for choice in (capi.KERNEL_VALU, capi.KERNEL_AUTO):
        with capi.Context(N, 1, I, D, nrot, True, ed, capi.QUADRATIC, capi.FLOAT, F, kernel_choice=choice) as ctx:
            ctx.set_som(som.reshape(N, -1))
            got.append(ctx.train(imgs) if train else ctx.map(imgs))
            if train:
                got[-1] = (ctx.get_som(), got[-1])
    (want, want_which), (out, which) = got
    lost = np.isnan(want)
    assert lost.any() or not train
    assert np.array_equal(np.isnan(out), lost) and np.array_equal(bits(out)[~lost], bits(want)[~lost])
    known = np.ones(want_which.shape, bool) if train else ~lost
    assert np.array_equal(which[known], want_which[known])


def test_memory_of_a_float_mapper_with_many_neurons():
    """A launch group's buffers stay within some 4 GiB, the lists of variants in question among them."""
    from test_zz_no_alloc import Hip
    hip = Hip()
    N, I, D, nrot, ed = 20000, 16, 12, 64, 6
    with capi.Context(9, 1, I, D, nrot, True, ed, capi.QUADRATIC, capi.FLOAT):
        before = hip.free_bytes()
        with capi.Context(N, 1, I, D, nrot, True, ed, capi.QUADRATIC, capi.FLOAT, max_batch=2048):
            taken = before - hip.free_bytes()
    say("bytes", taken)
    assert taken < 5 << 30


def _nearly_round(rng, n, C_, I, scale, noise=1e-3):
    """Images whose rotated copies differ by a thousandth: every variant's distance is close to every other's."""
    x = np.linspace(-1, 1, I)
    r2 = (x[:, None] ** 2 + x[None, :] ** 2) * rng.uniform(0.5, 3.0, (n, C_, 1, 1))
    return (scale * (np.exp(-r2) + noise * rng.random((n, C_, I, I)))).astype(np.float32)


@pytest.mark.parametrize("scale", [1e-20, 1e-19, 3e-19, 1e-18, 3e-18, 1e-15, 1.0, 1e15])
def test_screening_keeps_the_closest_variant_at_every_scale(scale):
    """The error of the rounded values is bounded by its measured size, whose squares are no float32 numbers any more where
    the values (fluxes in physical units) are below about 1e-18."""
    say("screening at scale", scale)
    N, I, D, nrot, ed, n = 60, 16, 12, 360, 5, 400
    rng = np.random.default_rng(17)
    som = (scale * rng.random((N, D * D))).astype(np.float32)
    imgs = _nearly_round(rng, n, 1, I, scale)
    want_heat, want_best = O.map_images(O.shape(N, 1, I, D, nrot, True, ed, capi.QUADRATIC, capi.FLOAT), som, imgs)
    with capi.Context(N, 1, I, D, nrot, True, ed, capi.QUADRATIC, capi.FLOAT) as ctx:
        ctx.set_som(som)
        heat, best = ctx.map(imgs)
    assert np.array_equal(best, want_best) and np.array_equal(bits(heat), bits(want_heat))


@pytest.mark.parametrize("ed_type", [capi.FLOAT, capi.UINT8, capi.UINT16])
def test_equal_distances_go_to_the_first_variant(ed_type):
    """A constant image has 720 identical quantised variants: every kernel must report variant 0 for every neuron
    (strict `<` over ascending variants, generate_euclidean_distance_matrix.h:43-50), also where the
    equal distances sit in different tiles of rotations."""
    N, C_, I, D, nrot, flip, ed = 9, 1, 32, 22, 360, True, 16
    rng = np.random.default_rng(17)
    som = rng.random((N, D * D), dtype=np.float32)
    imgs = np.full((2, C_, I, I), 0.5, np.float32)
    imgs[1, 0, 8:24, 8:24] = 0.25                     # constant inside every rotated region, not outside
    s = O.shape(N, C_, I, D, nrot, flip, ed, O.QUADRATIC, ed_type)
    oheat, obest = O.map_images(s, som, imgs)
    if ed_type != capi.FLOAT:                          # (in float32 the interpolation weights do not sum to exactly 1)
        assert (obest[0] == 0).all()
    choices = [capi.KERNEL_AUTO] if ed_type == capi.FLOAT else [capi.KERNEL_AUTO, capi.KERNEL_VALU, capi.KERNEL_MFMA_GEMM]
    if ed_type == capi.UINT8:
        choices += [capi.KERNEL_MFMA, capi.KERNEL_MFMA_SYM]
    for choice in choices:
        say("ties", ed_type, choice)
        with capi.Context(N, C_, I, D, nrot, flip, ed, capi.QUADRATIC, ed_type, kernel_choice=choice) as ctx:
            ctx.set_som(som)
            heat, best = ctx.map(imgs)
        assert np.array_equal(best, obest), choice
        assert np.array_equal(bits(heat), bits(oheat)), choice


@pytest.mark.parametrize("ed", [32, 45])
def test_largest_distances_do_not_lose_to_padding(ed):
    """Neurons of zeros against images of ones (and the reverse) give the largest distances a region
    allows: they must still beat the padded rows and columns of every integer kernel (ed = 45, 2025
    elements, takes the wide form of the symmetric kernel)."""
    N, C_, I, D, nrot, flip = 6, 1, 64, (44 if ed == 32 else 91), 360, True
    rng = np.random.default_rng(ed)
    som = rng.random((N, D * D), dtype=np.float32)
    som[0] = 0.0
    som[1] = 1.0
    imgs = rng.random((4, C_, I, I), dtype=np.float32)
    imgs[0] = 1.0
    imgs[1] = 0.0
    for ed_type in (capi.UINT8, capi.UINT16):
        s = O.shape(N, C_, I, D, nrot, flip, ed, O.QUADRATIC, ed_type)
        oheat, obest = O.map_images(s, som, imgs)
        choices = [capi.KERNEL_AUTO, capi.KERNEL_MFMA_GEMM] + ([capi.KERNEL_MFMA_SYM, capi.KERNEL_MFMA] if ed_type == capi.UINT8 else [])
        for choice in choices:
            say("extremes", ed, ed_type, choice)
            try:
                ctx = capi.Context(N, C_, I, D, nrot, flip, ed, capi.QUADRATIC, ed_type, kernel_choice=choice)
            except capi.PinkError:
                assert choice == capi.KERNEL_MFMA
                continue
            with ctx:
                ctx.set_som(som)
                heat, best = ctx.map(imgs)
            assert np.array_equal(bits(heat), bits(oheat)), (ed_type, choice)
            assert np.array_equal(best, obest), (ed_type, choice)


FUSED_TRAIN_SHAPES = [
    # N, C, I, D, nrot, flip, ed, shape, ed_type, images  -- operand packing inside the rotation and update kernels
    (10, 1, 20, 16, 24, True, 11, capi.CIRCULAR, capi.UINT16, 5),
    (70, 1, 20, 14, 8, False, 14, capi.QUADRATIC, capi.UINT8, 6),     # two column tiles, no flip
    (6, 3, 12, 10, 8, True, 6, capi.QUADRATIC, capi.UINT8, 4),        # three channels: their base rotations side by side in LDS, byte planes packed by the rotation kernel
    (6, 3, 12, 10, 8, True, 6, capi.QUADRATIC, capi.FLOAT, 4),        # three channels, float32 rows from the rotation kernel
    (5, 2, 9, 8, 4, True, 7, capi.CIRCULAR, capi.FLOAT, 3),           # region repeats channel 0 (CPU rule): no inverse table
    (5, 2, 9, 8, 4, True, 7, capi.CIRCULAR, capi.UINT16, 3),
    (4, 1, 200, 150, 8, True, 100, capi.CIRCULAR, capi.UINT8, 2),     # a large LDS tile in the rotation kernel
    (3, 1, 160, 129, 4, True, 128, capi.QUADRATIC, capi.FLOAT, 2),
    (4, 1, 290, 205, 8, True, 100, capi.CIRCULAR, capi.UINT8, 2),     # neurons too large for the rotation kernel's LDS tile
    (3, 1, 280, 201, 4, True, 128, capi.QUADRATIC, capi.FLOAT, 2),
    (4, 1, 160, 226, 8, True, 113, capi.QUADRATIC, capi.UINT8, 2),    # ... but the image fits: interpolated out of LDS
    (3, 1, 160, 226, 8, True, 113, capi.CIRCULAR, capi.UINT16, 2),
    (3, 1, 150, 201, 8, True, 100, capi.QUADRATIC, capi.FLOAT, 2),
    (3, 1, 210, 260, 8, True, 130, capi.QUADRATIC, capi.UINT8, 2),    # nothing in LDS and neurons larger than the image:
    (3, 1, 210, 297, 16, True, 148, capi.CIRCULAR, capi.FLOAT, 2),    # tiles of the base rotation that lie beyond the image
    (2, 2, 204, 230, 4, False, 100, capi.QUADRATIC, capi.UINT16, 2),
    (3, 1, 150, 200, 4, True, 200, capi.QUADRATIC, capi.UINT8, 2),    # 40 000 region elements: uint8 sums beyond 31 bits
    (2, 1, 150, 200, 4, False, 190, capi.QUADRATIC, capi.UINT16, 2),
    (2, 1, 100, 257, 4, False, 257, capi.QUADRATIC, capi.UINT8, 2),   # 66 049: beyond the matrix-core path's row length
    (2, 1, 100, 256, 4, False, 256, capi.QUADRATIC, capi.UINT16, 2),  # 65 536 (uint16 sums reach 2^48 just above that)
    (12, 1, 64, 44, 360, True, 32, capi.QUADRATIC, capi.UINT16, 2),   # 720 variants, uint16 planes out of the rotation kernel
    (70, 1, 40, 48, 36, True, 44, capi.QUADRATIC, capi.UINT16, 3),    # long rows, few tiles: 32 x 32 tiles (3 x 3 real ones among 16), each finished by its block
    (70, 1, 40, 52, 36, True, 48, capi.QUADRATIC, capi.UINT8, 3),     # the same for uint8 (72 k-steps)
    # small uint8 trainers: distance, best match and update of an image in one launch
    (33, 1, 44, 40, 4, True, 40, capi.QUADRATIC, capi.UINT8, 5),      # 1600 elements per neuron, 50 k-steps (two batches of operand loads), a second column tile of one neuron
    (64, 1, 30, 28, 16, True, 20, capi.CIRCULAR, capi.UINT8, 5),      # 32 variants (a full row tile), eight stored variants staged in LDS
    (5, 2, 14, 12, 1, True, 9, capi.QUADRATIC, capi.UINT8, 4),        # one rotation and its flip, two channels
    (7, 1, 14, 12, 1, False, 9, capi.QUADRATIC, capi.UINT8, 3),       # a single variant
    (40, 1, 20, 20, 8, True, 20, capi.QUADRATIC, capi.UINT8, 7),      # an odd number of images: the SOM operand ends in its second buffer
    # small float32 trainers: the distance launch of an image applies the update of the image before it
    (70, 1, 20, 14, 32, True, 9, capi.CIRCULAR, capi.FLOAT, 5),       # three chunks of 64 elements, neurons not a multiple of four
    (9, 1, 12, 8, 16, True, 8, capi.QUADRATIC, capi.FLOAT, 4),        # a single chunk
    (130, 2, 16, 11, 4, True, 11, capi.QUADRATIC, capi.FLOAT, 3),     # two channels, three keys per lane in the search
    (256, 1, 14, 10, 8, False, 10, capi.QUADRATIC, capi.FLOAT, 3),    # the most neurons that train this way
    (257, 1, 14, 10, 8, False, 10, capi.QUADRATIC, capi.FLOAT, 3),    # ... and one more
    (103, 1, 20, 14, 360, True, 12, capi.QUADRATIC, capi.FLOAT, 3),   # 12 x 26 blocks of four neurons are more than the CUs: five per block, the last block three
    (110, 1, 20, 14, 360, True, 9, capi.CIRCULAR, capi.FLOAT, 3),     # ... six per block
    (131, 1, 20, 14, 360, True, 9, capi.QUADRATIC, capi.FLOAT, 3),    # ... seven, three keys per lane in the search
    (165, 1, 20, 14, 360, True, 12, capi.QUADRATIC, capi.FLOAT, 4),   # ... eight, the last block five
]


@pytest.mark.parametrize("N,C_,I,D,nrot,flip,ed,shape_,ed_type,n", FUSED_TRAIN_SHAPES)
def test_train_over_shapes(N, C_, I, D, nrot, flip, ed, shape_, ed_type, n):
    say("train shapes", N, C_, I, D, nrot, flip, ed, shape_, ed_type, n)
    rng = np.random.default_rng(N + I * 3 + nrot)
    som0 = rng.random((N, C_ * D * D), dtype=np.float32)
    imgs = rng.random((n, C_, I, I), dtype=np.float32)
    F = capi.make_update_factors(capi.CARTESIAN, [N], capi.GAUSSIAN, 1.0, 0.5)
    F[F < 0.01] = 0.0                                        # some neurons are skipped by the update
    s = O.shape(N, C_, I, D, nrot, flip, ed, shape_, ed_type)
    want = som0.copy()
    obmu = O.train(s, want, imgs, F)
    with capi.Context(N, C_, I, D, nrot, flip, ed, shape_, ed_type, F, max_batch=2) as ctx:
        ctx.set_som(som0)
        bmu = np.concatenate([ctx.train(imgs[:1]), ctx.train(imgs[1:])])      # two calls, groups of two images
        som = ctx.get_som()
        # the packed operand the update kernel maintains must match a fresh pack of the same weights
        d1, ssd1, best1 = ctx.distance(imgs[0])
        ctx.set_som(som)
        d2, ssd2, best2 = ctx.distance(imgs[0])
    assert np.array_equal(bmu, obmu)
    assert np.array_equal(bits(som), bits(want))             # gate 1e-4; achieved and asserted: bit-exact
    assert np.array_equal(bits(d1), bits(d2)) and np.array_equal(ssd1, ssd2) and np.array_equal(best1, best2)


SMALL_UINT8_SHAPES = [s for s in FUSED_TRAIN_SHAPES if s[8] == capi.UINT8 and s[0] <= 64 and s[4] * (2 if s[5] else 1) <= 32
                      and s[1] * s[3] * s[3] <= 2048] + [
    (64, 1, 28, 28, 4, True, 28, capi.QUADRATIC, capi.UINT8, 40),     # the 8 x 8 MNIST-sized trainer of the benchmark set
    (1, 1, 16, 16, 4, True, 12, capi.QUADRATIC, capi.UINT8, 9),       # one neuron: an exchange with itself
    (64, 1, 45, 45, 4, False, 45, capi.QUADRATIC, capi.UINT8, 6),     # 2025 elements: four per thread, 64 k-steps
    (9, 1, 32, 32, 4, True, 31, capi.QUADRATIC, capi.UINT8, 6),       # 961: sixteen 64-byte k-steps of a tile
    (5, 1, 22, 22, 16, True, 22, capi.CIRCULAR, capi.UINT8, 6),       # two tiles: six,
    (5, 1, 29, 28, 16, True, 27, capi.QUADRATIC, capi.UINT8, 6),      # twelve,
    (5, 1, 32, 32, 16, True, 32, capi.QUADRATIC, capi.UINT8, 6),      # sixteen
    (4, 1, 20, 20, 20, False, 19, capi.QUADRATIC, capi.UINT8, 6),     # the second with four rows
    (3, 1, 33, 33, 4, True, 33, capi.QUADRATIC, capi.UINT8, 5),       # 1089 elements: one tile
    (4, 1, 36, 36, 12, True, 36, capi.QUADRATIC, capi.UINT8, 5),      # 1296 and two tiles: eight waves
]


@pytest.mark.parametrize("form", ["resident", "gives up", "off", "tags wrap"])
@pytest.mark.parametrize("N,C_,I,D,nrot,flip,ed,shape_,ed_type,n", SMALL_UINT8_SHAPES)
def test_small_uint8_trainer_forms(monkeypatch, N, C_, I, D, nrot, flip, ed, shape_, ed_type, n, form):
    """Small uint8 trainers run a whole launch group in one resident launch whose blocks exchange a word per image;
    when a block gives up waiting for the others (forced here by a wait limit of zero polls: every kernel still
    ends by itself) nothing of the context has changed and the group is trained again with one launch per image,
    as it is with the resident form switched off.  All against the oracle, bit for bit."""
    say("small uint8 trainer", form, N, C_, I, D, nrot, flip, ed, shape_, n)
    if form == "gives up":
        monkeypatch.setenv("PINK_HIP_RESIDENT_SPIN_LIMIT", "0")
    if form == "off":
        monkeypatch.setenv("PINK_HIP_RESIDENT_TRAINER", "0")
    if form == "tags wrap":
        # the exchange tags every image with a running 32-bit number; start it where the second call passes the end
        monkeypatch.setenv("PINK_HIP_RESIDENT_FIRST_TAG", str(0xfffffff0 - n + 1))
    rng = np.random.default_rng(N * 7 + I + nrot)
    som0 = rng.random((N, C_ * D * D), dtype=np.float32)
    imgs = rng.random((n, C_, I, I), dtype=np.float32)
    F = capi.make_update_factors(capi.CARTESIAN, [N], capi.GAUSSIAN, 1.0, 0.5)
    F[F < 0.01] = 0.0
    s = O.shape(N, C_, I, D, nrot, flip, ed, shape_, ed_type)
    want = som0.copy()
    obmu = O.train(s, want, imgs, F)
    for max_batch in (0, 3):                                 # the whole call in one group; groups of three images
        with capi.Context(N, C_, I, D, nrot, flip, ed, shape_, ed_type, F, max_batch=max_batch) as ctx:
            ctx.set_som(som0)
            bmu = np.concatenate([ctx.train(imgs[:2]), ctx.train(imgs[2:])])
            som = ctx.get_som()
            counts = ctx.update_counts()
            d1, ssd1, best1 = ctx.distance(imgs[0])          # the operand and norms the trainer left behind
            ctx.set_som(som)
            d2, ssd2, best2 = ctx.distance(imgs[0])
        assert np.array_equal(bmu, obmu), max_batch
        assert np.array_equal(bits(som), bits(want)), max_batch
        assert np.array_equal(counts, np.bincount(obmu, minlength=N)), max_batch
        assert np.array_equal(bits(d1), bits(d2)) and np.array_equal(ssd1, ssd2) and np.array_equal(best1, best2)


RESIDENT_SYMMETRIC_SHAPES = [
    (3, 1, 9, 9, 1, False, 7, capi.QUADRATIC, capi.UINT8, 5),          # one variant
    (1, 1, 16, 16, 4, True, 12, capi.QUADRATIC, capi.UINT16, 5),       # one neuron, one base rotation: k cut seven ways
    (7, 1, 16, 16, 4, True, 11, capi.CIRCULAR, capi.UINT16, 6),        # symmetries that cover different elements
    (9, 1, 20, 14, 68, True, 9, capi.QUADRATIC, capi.UINT16, 5),       # 17 base rotations: two tiles, k cut three ways
    (6, 2, 18, 12, 132, True, 8, capi.QUADRATIC, capi.UINT8, 4),       # 33: three tiles; two channels
    (5, 1, 24, 33, 200, False, 31, capi.CIRCULAR, capi.UINT8, 4),      # 50: four tiles
    (4, 1, 14, 10, 456, True, 7, capi.QUADRATIC, capi.UINT16, 3),      # 114: eight tiles for seven waves
    (3, 1, 60, 64, 40, True, 60, capi.QUADRATIC, capi.UINT8, 3),       # ten elements per thread
    (2, 1, 100, 100, 24, True, 97, capi.QUADRATIC, capi.UINT16, 2),    # 24
    (257, 1, 12, 8, 20, True, 6, capi.QUADRATIC, capi.UINT8, 4),       # two neurons per block, the last block with one
    (260, 1, 40, 36, 12, True, 36, capi.QUADRATIC, capi.UINT16, 3),
    (520, 1, 12, 10, 20, True, 8, capi.CIRCULAR, capi.UINT16, 3),      # four neurons per block
    (601, 1, 30, 28, 8, True, 28, capi.QUADRATIC, capi.UINT8, 3),
    (2, 1, 208, 40, 60, True, 20, capi.QUADRATIC, capi.UINT8, 2),      # an image larger than the LDS
    (3, 1, 22, 22, 1, False, 20, capi.QUADRATIC, capi.FLOAT, 5),
    (1, 1, 24, 24, 4, True, 22, capi.QUADRATIC, capi.FLOAT, 5),
    (7, 1, 26, 26, 4, True, 25, capi.CIRCULAR, capi.FLOAT, 6),
    (9, 1, 30, 24, 68, True, 21, capi.QUADRATIC, capi.FLOAT, 5),
    (6, 2, 26, 18, 132, True, 15, capi.QUADRATIC, capi.FLOAT, 4),
    (5, 1, 24, 33, 200, False, 31, capi.CIRCULAR, capi.FLOAT, 4),
    (4, 1, 30, 28, 448, True, 23, capi.QUADRATIC, capi.FLOAT, 3),      # seven tiles, the most
    (3, 1, 60, 64, 40, True, 60, capi.QUADRATIC, capi.FLOAT, 3),       # runs in four blocks, three waves sum
    (300, 1, 16, 12, 208, True, 11, capi.QUADRATIC, capi.FLOAT, 4),
    (260, 1, 40, 36, 12, True, 33, capi.QUADRATIC, capi.FLOAT, 3),
    (520, 1, 30, 26, 20, True, 25, capi.CIRCULAR, capi.FLOAT, 3),
    (2, 1, 208, 40, 60, True, 20, capi.QUADRATIC, capi.FLOAT, 2),
]


@pytest.mark.parametrize("form", ["resident", "gives up", "tags wrap"])
@pytest.mark.parametrize("N,C_,I,D,nrot,flip,ed,shape_,ed_type,n", RESIDENT_SYMMETRIC_SHAPES)
def test_resident_symmetric_trainer_forms(monkeypatch, N, C_, I, D, nrot, flip, ed, shape_, ed_type, n, form):
    """Trainers with the symmetries on the SOM side keep their neurons on the device over a launch group (see
    test_small_uint8_trainer_forms for the exchange between the blocks).  What a launch that gives up leaves undone, and the groups
    queued behind it, the launch that follows it trains; the next call takes the other form."""
    say("resident symmetric trainer", form, N, C_, I, D, nrot, flip, ed, shape_, ed_type, n)
    if form == "gives up":
        monkeypatch.setenv("PINK_HIP_RESIDENT_SPIN_LIMIT", "0")
    if form == "tags wrap":
        monkeypatch.setenv("PINK_HIP_RESIDENT_FIRST_TAG", str(0xfffe - n + 2))      # 16-bit tags: 0xfffe is the last
    rng = np.random.default_rng(N * 5 + I + nrot)
    som0 = rng.random((N, C_ * D * D), dtype=np.float32)
    imgs = rng.random((n, C_, I, I), dtype=np.float32)
    F = capi.make_update_factors(capi.CARTESIAN, [N], capi.GAUSSIAN, 1.0, 0.5)
    F[F < 0.01] = 0.0
    s = O.shape(N, C_, I, D, nrot, flip, ed, shape_, ed_type)
    want = som0.copy()
    obmu = O.train(s, want, imgs, F)
    for max_batch, first in ((0, 1), (2, 1), (1, n)):
        with capi.Context(N, C_, I, D, nrot, flip, ed, shape_, ed_type, F, max_batch=max_batch) as ctx:
            ctx.set_som(som0)
            bmu = ctx.train(imgs[:first])
            if first < n:
                bmu = np.concatenate([bmu, ctx.train(imgs[first:])])
            som = ctx.get_som()
            counts = ctx.update_counts()
            d1, ssd1, best1 = ctx.distance(imgs[0])
            ctx.set_som(som)
            d2, ssd2, best2 = ctx.distance(imgs[0])
        assert np.array_equal(bmu, obmu), max_batch
        assert np.array_equal(bits(som), bits(want)), max_batch
        assert np.array_equal(counts, np.bincount(obmu, minlength=N)), max_batch
        assert np.array_equal(bits(d1), bits(d2)) and np.array_equal(ssd1, ssd2) and np.array_equal(best1, best2)


# (neurons of a block x blocks that share out an image's rows; tiles of a wave; chunks of 64 orbits of a neuron, of a wave)
RESIDENT_INTEGER_PLANS = [
    (90, 1, 40, 40, 360, True, 34, capi.QUADRATIC, capi.UINT8, 3),       # 2 x 3, two groups of waves
    (91, 1, 40, 40, 360, True, 35, capi.QUADRATIC, capi.UINT16, 3),      # the last block holds one neuron; an odd region in an even neuron
    (130, 1, 30, 30, 360, True, 21, capi.QUADRATIC, capi.UINT8, 3),      # 1 x 1, two groups of waves, three tiles to a wave
    (331, 1, 60, 60, 240, True, 55, capi.CIRCULAR, capi.UINT16, 2),      # 2 x 1, four groups of waves
    (331, 1, 90, 80, 360, True, 75, capi.CIRCULAR, capi.UINT16, 2),      # 4 x 3: nine chunks of a neuron, up to six of a wave
    (60, 2, 36, 36, 500, True, 24, capi.QUADRATIC, capi.UINT16, 3),      # 2 x 4
    (5, 1, 20, 20, 1000, True, 15, capi.QUADRATIC, capi.UINT16, 3),      # 1 x 4, four tiles each; 250 rotations are not whole tiles
    (4, 1, 24, 24, 2400, True, 19, capi.QUADRATIC, capi.UINT16, 2),      # 1 x 5, eight groups of waves
    (255, 1, 30, 30, 720, False, 20, capi.CIRCULAR, capi.UINT8, 3),      # twelve tiles, four groups of waves
    (10, 1, 100, 100, 200, True, 91, capi.QUADRATIC, capi.UINT8, 2),     # 1 x 4, seventeen chunks
    (12, 1, 100, 100, 80, False, 98, capi.QUADRATIC, capi.UINT16, 2),
    (200, 1, 120, 120, 24, True, 98, capi.QUADRATIC, capi.UINT8, 2),     # twenty chunks
    (6, 1, 150, 150, 40, True, 146, capi.QUADRATIC, capi.UINT8, 2),      # 43 chunks
    (6, 1, 150, 150, 40, True, 143, capi.QUADRATIC, capi.UINT8, 2),      # 42, six to a wave
    (513, 1, 60, 60, 24, True, 50, capi.QUADRATIC, capi.UINT8, 2),       # 3 x 1
    (625, 1, 34, 34, 360, True, 24, capi.QUADRATIC, capi.UINT8, 2),      # ... three tiles to a wave
    (331, 1, 90, 90, 360, True, 64, capi.QUADRATIC, capi.UINT8, 2),      # 3 x 2, the last block holds one neuron
    (1023, 1, 20, 18, 12, True, 17, capi.QUADRATIC, capi.UINT16, 3),     # 4 x 1, the last block holds three
    (40, 1, 23, 22, 36, True, 22, capi.QUADRATIC, capi.UINT16, 3),       # 66 orbits: a chunk and two more
    (40, 1, 23, 21, 36, True, 21, capi.QUADRATIC, capi.UINT8, 3),        # an odd neuron: the middle twice
    (12, 1, 30, 70, 80, True, 60, capi.QUADRATIC, capi.UINT8, 3),        # places that no rotation of the image reaches: three of eight chunks
    (500, 1, 30, 71, 40, True, 61, capi.CIRCULAR, capi.UINT16, 3),
    (400, 1, 20, 60, 24, False, 49, capi.QUADRATIC, capi.UINT16, 2),
    (9, 1, 64, 200, 48, True, 181, capi.QUADRATIC, capi.UINT8, 2),       # ten chunks to a thread
    (9, 1, 64, 200, 48, True, 180, capi.QUADRATIC, capi.UINT16, 2),
    (3, 1, 40, 190, 16, True, 186, capi.QUADRATIC, capi.UINT16, 2),      # all of them: saturated, their squares could pass 2^31
    (60, 1, 100, 140, 36, True, 130, capi.QUADRATIC, capi.UINT8, 2),     # 34 chunks, 31 reached
    (8, 2, 61, 40, 68, True, 25, capi.QUADRATIC, capi.UINT16, 3),        # a window of the image; a region that symmetries move by a pixel
    (8, 1, 5, 9, 12, True, 8, capi.QUADRATIC, capi.UINT8, 3),            # an image smaller than its window; one piece of most rows
    (8, 1, 200, 64, 40, False, 37, capi.CIRCULAR, capi.UINT8, 3),
]


@pytest.mark.parametrize("form", ["resident", "gives up", "tags wrap"])
@pytest.mark.parametrize("N,C_,I,D,nrot,flip,ed,shape_,ed_type,n", RESIDENT_INTEGER_PLANS)
def test_resident_integer_trainer_plans(monkeypatch, N, C_, I, D, nrot, flip, ed, shape_, ed_type, n, form):
    """How the neurons and an image's rows are dealt to the blocks, at the edges of chunks, tiles, groups of waves and blocks."""
    test_resident_symmetric_trainer_forms(monkeypatch, N, C_, I, D, nrot, flip, ed, shape_, ed_type, n, form)


def awkward(kind, rng, som, imgs):
    """Values that the integer conversions send to the ends of their range, in images and in the weights of the middle of a neuron; in place."""
    if kind == "outside":
        som *= 4
        som -= 1.5
        imgs *= 4
        imgs -= 1.5
        return
    for a in (som, imgs):
        mid = a.shape[-1] // 2
        for value in {"infinite": (np.inf, -np.inf), "nan": (np.nan, -np.nan), "saturated": ()}[kind]:
            picked = rng.integers(0, a.shape[0], 2)
            a[picked, ..., mid + rng.integers(-2, 3, 2), mid + rng.integers(-2, 3, 2)] = value
    if kind == "saturated":                                            # (squares as large as they can be, but the closest neuron's)
        som[1:] = 1.0 + 1e20 * som[1:]
        som[0] = 0.9


AWKWARD_INTEGER_TRAINERS = [(kind,) + shape for kind in ("outside", "infinite", "nan") for shape in (
    (9, 1, 28, 28, 4, True, 28, capi.QUADRATIC, capi.UINT8, 6),        # eight symmetries, one wave multiplies
    (20, 1, 24, 18, 40, True, 16, capi.QUADRATIC, capi.UINT8, 6),
    (20, 1, 24, 18, 40, True, 16, capi.CIRCULAR, capi.UINT16, 6),
    (300, 1, 16, 12, 68, True, 11, capi.QUADRATIC, capi.UINT16, 4),    # two neurons to a block
    (9, 1, 64, 200, 48, True, 181, capi.QUADRATIC, capi.UINT8, 2),     # ten orbits a thread, places that no rotation reaches
    (9, 1, 64, 200, 48, True, 180, capi.QUADRATIC, capi.UINT16, 2),
)] + [("saturated",) + shape for shape in (
    (3, 1, 40, 190, 16, True, 186, capi.QUADRATIC, capi.UINT8, 2),     # unreached squares up to 2.2e9 beside reached ones: past 2^31
    (3, 1, 40, 190, 16, True, 181, capi.QUADRATIC, capi.UINT16, 2),    # ... up to 32 761 times 255^2 in each of three sums: just below it
    (3, 1, 40, 190, 16, True, 186, capi.QUADRATIC, capi.UINT16, 2),    # they would pass it: all places are taken for reached
)]


@pytest.mark.parametrize("form", ["resident", "gives up", "off"])
@pytest.mark.parametrize("kind,N,C_,I,D,nrot,flip,ed,shape_,ed_type,n", AWKWARD_INTEGER_TRAINERS)
def test_integer_trainers_on_awkward_values(monkeypatch, kind, N, C_, I, D, nrot, flip, ed, shape_, ed_type, n, form):
    """Values outside [0, 1], infinite ones and none at all quantise to the ends of the range (no number: 0) in every form of a trainer."""
    say("awkward integer trainer", kind, form, N, C_, I, D, nrot, flip, ed, shape_, ed_type, n)
    if form == "gives up":
        monkeypatch.setenv("PINK_HIP_RESIDENT_SPIN_LIMIT", "0")
    if form == "off":
        monkeypatch.setenv("PINK_HIP_RESIDENT_TRAINER", "0")
    rng = np.random.default_rng(N + I + nrot)
    som0, imgs = rng.random((N, C_, D, D), dtype=np.float32), rng.random((n, C_, I, I), dtype=np.float32)
    awkward(kind, rng, som0, imgs)
    som0 = som0.reshape(N, -1)
    F = capi.make_update_factors(capi.CARTESIAN, [N], capi.GAUSSIAN, 1.0, 0.5)
    F[F < 0.01] = 0.0
    want = som0.copy()
    obmu = O.train(O.shape(N, C_, I, D, nrot, flip, ed, shape_, ed_type), want, imgs, F)
    lost = np.isnan(want)
    with capi.Context(N, C_, I, D, nrot, flip, ed, shape_, ed_type, F) as ctx:
        ctx.set_som(som0)
        bmu = np.concatenate([ctx.train(imgs[:1]), ctx.train(imgs[1:])])
        som = ctx.get_som()
    assert np.array_equal(bmu, obmu)
    assert np.array_equal(np.isnan(som), lost) and np.array_equal(bits(som)[~lost], bits(want)[~lost])


def test_resident_integer_trainer_of_the_most_rotations():
    """A group's operand is counted in 32 bits: an image's is 272 MB here, so seven make a group, where there were always eight."""
    N, I, nrot, n = 4, 90, 65536, 8
    say("resident integer trainer, 65536 rotations")
    rng = np.random.default_rng(3)
    som0, imgs = rng.random((N, I * I), dtype=np.float32), rng.random((n, I * I), dtype=np.float32)
    F = capi.make_update_factors(capi.CARTESIAN, [N], capi.GAUSSIAN, 1.0, 0.5)
    want = som0.copy()
    obmu = O.train(O.shape(N, 1, I, I, nrot, False, I, capi.QUADRATIC, capi.UINT16), want, imgs, F)
    with capi.Context(N, 1, I, I, nrot, False, I, capi.QUADRATIC, capi.UINT16, F) as ctx:
        ctx.set_som(som0)
        bmu, som = ctx.train(imgs), ctx.get_som()
    assert np.array_equal(bmu, obmu) and np.array_equal(bits(som).ravel(), bits(want).ravel())


@pytest.mark.parametrize("kind", ["outside", "infinite", "nan"])
@pytest.mark.parametrize("N,C_,I,D,nrot,flip,ed,shape_,ed_type,n", [
    (20, 1, 24, 18, 40, True, 16, capi.QUADRATIC, capi.UINT16, 6),
    (5, 1, 250, 64, 40, False, 37, capi.CIRCULAR, capi.UINT8, 4),      # uint8 beyond the other product's images,
    (3, 1, 180, 254, 8, True, 181, capi.QUADRATIC, capi.UINT8, 3),     # ... and regions
])
def test_orbit_mappers_on_awkward_values(N, C_, I, D, nrot, flip, ed, shape_, ed_type, n, kind):
    say("awkward integer mapper", kind, N, C_, I, D, nrot, flip, ed, shape_, ed_type, n)
    rng = np.random.default_rng(N + I + nrot)
    som, imgs = rng.random((N, C_, D, D), dtype=np.float32), rng.random((n, C_, I, I), dtype=np.float32)
    awkward(kind, rng, som, imgs)
    oheat, obest = O.map_images(O.shape(N, C_, I, D, nrot, flip, ed, shape_, ed_type), som, imgs)
    with capi.Context(N, C_, I, D, nrot, flip, ed, shape_, ed_type) as ctx:
        ctx.set_som(som.reshape(N, -1))
        heat, best = ctx.map(imgs)
    assert np.array_equal(bits(heat), bits(oheat)) and np.array_equal(best, obest)


@pytest.mark.parametrize("kind", ["blank", "flat", "alike", "zero", "nan", "grown", "faint", "flux"])
def test_resident_float_trainer_on_awkward_data(kind):
    """Images and weights that leave many variants or several neurons to the float32 sums."""
    say("resident float trainer", kind)
    N, C_, I, D, nrot, ed, n = 12, 1, 40, 32, 180, 25, 50
    rng = np.random.default_rng(5)
    som0, imgs = rng.random((N, C_ * D * D), dtype=np.float32), rng.random((n, C_, I, I), dtype=np.float32)
    F = capi.make_update_factors(capi.CARTESIAN, [N], capi.MEXICAN_HAT if kind == "grown" else capi.GAUSSIAN, 1.0, 0.5)
    if kind == "blank":
        imgs[1::3] = 0.0
    elif kind == "flat":
        imgs[2:] = 0.25                                                # (all variants alike, image after image)
    elif kind == "alike":
        som0[3:9] = som0[3]                                            # (neurons that tie)
    elif kind == "zero":
        som0[:] = 0.0
    elif kind == "nan":
        imgs[4, 0, I // 2, I // 2] = np.nan
    elif kind == "grown":
        som0[::5] *= 3000.0
    elif kind == "faint":
        imgs *= np.float32(0.003)                                      # (the product's error is the smaller one)
    elif kind == "flux":
        imgs, som0 = imgs * np.float32(2e-20), som0 * np.float32(5e-19)       # (squares that are no float32 numbers)
    s = O.shape(N, C_, I, D, nrot, True, ed, capi.QUADRATIC, capi.FLOAT)
    want = som0.copy()
    want_bmu = O.train(s, want, imgs, F)
    if kind == "nan":       # (no order among such distances: the kernel that sums every variant is the measure)
        with capi.Context(N, C_, I, D, nrot, True, ed, capi.QUADRATIC, capi.FLOAT, F, kernel_choice=capi.KERNEL_VALU) as ctx:
            ctx.set_som(som0)
            want_bmu, want = ctx.train(imgs), ctx.get_som()
    lost = np.isnan(want)
    assert lost.any() == (kind == "nan")
    with capi.Context(N, C_, I, D, nrot, True, ed, capi.QUADRATIC, capi.FLOAT, F) as ctx:
        ctx.set_som(som0)
        bmu = np.concatenate([ctx.train(imgs[:1]), ctx.train(imgs[1:])])
        som = ctx.get_som()
    assert np.array_equal(bmu, want_bmu) and np.array_equal(np.isnan(som), lost) and np.array_equal(bits(som)[~lost], bits(want)[~lost])


@pytest.mark.parametrize("kind", ["flat", "alike", "infinite image", "infinite weights", "nan", "grown"])
@pytest.mark.parametrize("N,I,D,nrot,ed,shape_", [
    (12, 40, 32, 180, 25, capi.QUADRATIC),
    (12, 60, 50, 100, 44, capi.CIRCULAR),                              # rows of more than 1024 places
    (150, 30, 25, 100, 22, capi.QUADRATIC),                            # more neurons than a request brings words of; not symmetric
    (300, 30, 26, 60, 21, capi.QUADRATIC),                             # two neurons to a block
    (520, 30, 26, 60, 25, capi.CIRCULAR),                              # four
])
def test_resident_float_trainer_on_awkward_data_over_shapes(N, I, D, nrot, ed, shape_, kind):
    """... in every form of the exchange: lists past their length, neurons of several blocks that tie, what is no number; against the
    kernel that sums every variant."""
    say("resident float trainer", kind, N, I, D, nrot, ed, shape_)
    n = 24
    rng = np.random.default_rng(N + D)
    som0, imgs = rng.random((N, D, D), dtype=np.float32), rng.random((n, 1, I, I), dtype=np.float32)
    F = capi.make_update_factors(capi.CARTESIAN, [N], capi.MEXICAN_HAT if kind == "grown" else capi.GAUSSIAN, 1.0, 0.5)
    if kind == "flat":
        imgs[1::3] = 0.25
    elif kind == "alike":
        som0[N // 4:N - 2] = som0[3]
        F[F < 0.01] = 0.0                                              # (most of them stay alike)
    elif kind == "infinite image":
        imgs[3, 0, I // 2, I // 2], imgs[9, 0, I // 2 - 3, I // 2] = np.inf, -np.inf
    elif kind == "infinite weights":
        som0[::5, D // 2, D // 2], som0[3::5, D // 2, D // 2 + 1] = np.inf, -np.inf
    elif kind == "nan":
        imgs[5, 0, I // 2, I // 2 + 2] = np.nan
    elif kind == "grown":
        som0[::5] *= 3000.0
    got = []
    for choice in (capi.KERNEL_VALU, capi.KERNEL_AUTO):
        with capi.Context(N, 1, I, D, nrot, True, ed, shape_, capi.FLOAT, F, kernel_choice=choice) as ctx:
            ctx.set_som(som0.reshape(N, -1))
            bmu = np.concatenate([ctx.train(imgs[:9]), ctx.train(imgs[9:])])
            got.append((bmu, ctx.get_som(), ctx.update_counts()))
    (want_bmu, want, want_counts), (bmu, som, counts) = got
    lost = np.isnan(want)
    assert lost.any() == (kind in ("infinite image", "infinite weights", "nan"))
    assert np.array_equal(bmu, want_bmu) and np.array_equal(counts, want_counts)
    assert np.array_equal(np.isnan(som), lost) and np.array_equal(bits(som)[~lost], bits(want)[~lost])


class FloatTrainer:
    """A resident float32 trainer beside one that sums every variant; counts the launch groups of a call."""
    def __init__(self, N=12, I=40, D=32, nrot=180, ed=25):
        self.N, self.I, self.D, self.nrot, self.ed = N, I, D, nrot, ed
        F = capi.make_update_factors(capi.CARTESIAN, [self.N], capi.GAUSSIAN, 1.0, 0.5)
        self.ctx, self.plain = (capi.Context(self.N, 1, self.I, self.D, self.nrot, True, self.ed, capi.QUADRATIC, capi.FLOAT, F, kernel_choice=k)
                                for k in (capi.KERNEL_AUTO, capi.KERNEL_VALU))
        self.rng = np.random.default_rng(5)
        som = self.rng.random((self.N, self.D ** 2), dtype=np.float32)
        for c in (self.ctx, self.plain):
            c.set_som(som)
        self.ctx.set_profiling(True)

    def images(self, n, flat=None):
        imgs = self.rng.random((n, 1, self.I, self.I), dtype=np.float32)
        if flat:
            imgs[flat] = 0.25                                          # (all variants alike)
        return imgs

    def groups(self, imgs, kernels="rotate"):
        before = self.ctx.kernel_times()[kernels][0]
        assert np.array_equal(self.ctx.train(imgs), self.plain.train(imgs))
        return self.ctx.kernel_times()[kernels][0] - before

    def check(self):
        assert np.array_equal(bits(self.ctx.get_som()), bits(self.plain.get_som()))
        assert np.array_equal(self.ctx.update_counts(), self.plain.update_counts())
        self.ctx.close()
        self.plain.close()


def test_resident_float_trainer_is_tried_on_enough_images():
    """One image that went through says little of the call behind it: flat images show within 32 of them, and the others take the
    other form, whose launch groups are smaller."""
    say("resident float trainer, one image first")
    t = FloatTrainer()
    assert t.groups(t.images(1)) == 1
    groups = t.groups(t.images(300, slice(None)))
    say("groups", groups)
    t.check()
    assert groups >= 6


def test_resident_float_trainer_looks_up_during_a_call():
    """A call that turns flat behind images that went through well leaves the resident form within a few groups."""
    say("resident float trainer, a long call turns flat")
    t = FloatTrainer()
    t.groups(t.images(64))
    groups = t.groups(t.images(3000, slice(300, None)))
    say("groups", groups)
    t.check()
    assert groups >= 30


def test_resident_float_trainer_leaves_what_is_slow_and_comes_back():
    """A launch that spent too many sums without giving up: the next 256 images take the other form, then the form is tried again."""
    say("resident float trainer, slow launches")
    t = FloatTrainer()
    t.groups(t.images(64))
    proven = t.groups(t.images(150))
    t.groups(t.images(90, slice(None, None, 3)))
    away, back = t.groups(t.images(256)), t.groups(t.images(150))
    say("groups", proven, away, back)
    t.check()
    assert proven == 1 and away >= 4 and back <= 2


def test_resident_float_trainer_forgets_slow_launches():
    """The images that take the other form behind a slow launch are four times as many the next time, but not where a thousand went
    through well between."""
    say("resident float trainer, slow launches long apart")
    t = FloatTrainer()
    slow = slice(None, None, 3)
    t.groups(t.images(64))
    for between in (0, 1200):
        t.groups(t.images(between))
        t.groups(t.images(90, slow))
        t.groups(t.images(256))
        back = t.groups(t.images(150))
        say("groups", back)
        assert back <= 2
    t.groups(t.images(90, slow))
    t.groups(t.images(256))
    still_away = t.groups(t.images(150))
    say("groups", still_away)
    t.check()
    assert still_away > 2


@pytest.mark.parametrize("N,I,D,nrot,ed", [(9, 136, 96, 360, 91), (100, 80, 56, 360, 51)])
def test_screened_float_trainer_leaves_flat_images_to_the_sums(monkeypatch, N, I, D, nrot, ed):
    """Images that keep every variant, one after the other, go through the kernel that sums every variant and updates on the way, without
    an update launch per image; images that do not are screened again after a while."""
    monkeypatch.setenv("PINK_HIP_RESIDENT_TRAINER", "0")
    say("screened float trainer, flat images", N, I, D, nrot, ed)
    t = FloatTrainer(N, I, D, nrot, ed)
    before = t.groups(t.images(60), "update")
    flat = [t.groups(t.images(60, slice(None)), "update") for _ in range(4)]
    away, back = t.groups(t.images(200), "update"), t.groups(t.images(150), "update")
    say("update launches", before, flat, away, back)
    t.check()
    assert before >= 60 and flat[-1] < 30 and away < 150 and back >= 100


@pytest.mark.parametrize("N,I,D,nrot,ed", [
    (12, 40, 32, 180, 25),
    (300, 30, 26, 60, 21),                                             # two neurons to a block
    (200, 60, 50, 100, 45),                                            # resident, screened and summed
    (9, 100, 96, 360, 91),                                             # screened and summed
    (100, 24, 20, 360, 15),
])
def test_float_trainer_in_calls_of_every_size(N, I, D, nrot, ed):
    """Calls of few images take a form of their own; every form goes on from the weights that another left."""
    say("float trainer in calls of every size", N, I, D, nrot, ed)
    t = FloatTrainer(N, I, D, nrot, ed)
    for n in (1, 1, 33, 1, 2, 40, 3, 4, 36, 1, 6, 12, 34, 34, 5):
        imgs = t.images(n)
        t.groups(imgs)
        if n < 34:
            (d, _, best), (want_d, _, want_best) = t.ctx.distance(imgs[0]), t.plain.distance(imgs[0])
            assert np.array_equal(best, want_best) and np.array_equal(bits(d), bits(want_d)), n
    t.check()


@pytest.mark.parametrize("N,I,D,nrot,ed", [(12, 40, 32, 180, 25), (9, 64, 51, 8, 45), (9, 180, 150, 8, 128)])
def test_float_training_of_one_image_takes_no_longer_than_its_kernels(monkeypatch, N, I, D, nrot, ed):
    """A call of one image: what sums every variant in a launch, not what launches a group or five kernels."""
    import time
    from test_zz_no_alloc import Hip
    F = capi.make_update_factors(capi.CARTESIAN, [N], capi.GAUSSIAN, 1.0, 0.5)
    hip = Hip()
    rng = np.random.default_rng(4)
    imgs, som = hip.upload(rng.random((40, 1, I, I), dtype=np.float32)), rng.random((N, D * D), dtype=np.float32)
    taken = []
    for choice in (capi.KERNEL_VALU, capi.KERNEL_AUTO):
        with capi.Context(N, 1, I, D, nrot, True, ed, capi.QUADRATIC, capi.FLOAT, F, kernel_choice=choice) as ctx:
            ctx.set_som(som)
            ctx.train_device(imgs, 40)
            times = []
            for _ in range(60):
                start = time.perf_counter()
                ctx.train_device(imgs, 1)
                ctx.synchronize()
                times.append(time.perf_counter() - start)
            taken.append(sorted(times)[30])
    hip.release()
    say("one image", taken)
    assert taken[1] < 1.2 * taken[0]


def test_resident_float_training_is_queued():
    """pink_hip_train_device returns while the device still trains a context's first images."""
    import time
    from test_zz_no_alloc import Hip
    N, I, D, n = 9, 64, 64, 32
    F = capi.make_update_factors(capi.CARTESIAN, [3, 3], capi.GAUSSIAN, 1.1, 0.2)
    hip = Hip()
    imgs, bmu = hip.upload(np.random.default_rng(4).random((n, 1, I, I), dtype=np.float32)), hip.alloc(4 * n)
    for _ in range(2):                                                 # (the first context loads the kernels)
        with capi.Context(N, 1, I, D, 360, True, 64, capi.QUADRATIC, capi.FLOAT, F) as ctx:
            ctx.set_som(np.random.default_rng(5).random((N, D * D), dtype=np.float32))
            start = time.perf_counter()
            ctx.train_device(imgs, n, bmu)
            queued = time.perf_counter() - start
            ctx.synchronize()
            whole = time.perf_counter() - start
    hip.release()
    say("queued after", queued, "of", whole)
    assert queued < 0.7 * whole


@pytest.mark.parametrize("N,I,D,nrot,ed,ed_type", [
    (30, 24, 30, 20, 9, capi.UINT8),
    (30, 24, 30, 20, 9, capi.UINT16),
    (30, 40, 35, 20, 21, capi.FLOAT),
    (3, 70, 110, 48, 95, capi.UINT16),                                 # (weights in orbit order)
    (30, 1, 9, 4, 5, capi.UINT8),                                      # images of one pixel
])
def test_factors_that_move_some_elements_only(N, I, D, nrot, ed, ed_type):
    """Elements outside the region are passed by where no element of a wave can move: factors down to nothing, small weights."""
    say("factors that move some elements", N, I, D, nrot, ed, ed_type)
    n = 6
    rng = np.random.default_rng(N + I)
    som0, imgs = rng.random((N, D * D), dtype=np.float32), rng.random((n, 1, I, I), dtype=np.float32)
    som0[1::3] += np.float32(0.5)                                      # (no small weights)
    som0[2::3, ::D] *= np.float32(1e-9)
    som0[::4, 5] = 0.0
    imgs[2] *= np.float32(-30.0)
    imgs[3] = 0.0
    F = capi.make_update_factors(capi.CARTESIAN, [N], capi.GAUSSIAN, 1.5, 0.5) ** np.float32(1.3)
    F[:, ::5] *= np.float32(3e-8)
    F[:, 1::7] *= np.float32(-1e-7)
    want = som0.copy()
    want_bmu = O.train(O.shape(N, 1, I, D, nrot, True, ed, capi.QUADRATIC, ed_type), want, imgs, F)
    with capi.Context(N, 1, I, D, nrot, True, ed, capi.QUADRATIC, ed_type, F) as ctx:
        ctx.set_som(som0)
        assert np.array_equal(ctx.train(imgs), want_bmu) and np.array_equal(bits(ctx.get_som()), bits(want))


@pytest.mark.parametrize("N,I,D,nrot,ed,ed_type,pixel", [
    (30, 24, 30, 20, 9, capi.UINT8, (1, 12)),
    (30, 40, 35, 20, 21, capi.FLOAT, (3, 20)),
    (3, 70, 110, 48, 95, capi.UINT16, None),                           # (weights in orbit order; no pixel beside the region)
])
def test_small_factors_on_weights_without_bounds(N, I, D, nrot, ed, ed_type, pixel):
    """inf - (inf - x) f is no number under the smallest factor, nor is a difference that overflows small: such weights outside the
    region are not passed by.  Factors of zero leave them."""
    say("small factors on weights without bounds", N, I, D, nrot, ed, ed_type)
    n = 5
    rng = np.random.default_rng(N + I)
    som0, imgs = rng.random((N, D, D), dtype=np.float32), rng.random((n, 1, I, I), dtype=np.float32)
    m = (D - ed) // 2
    outside = np.ones((D, D), bool)
    outside[m:m + ed, m:m + ed] = False
    for k, value in enumerate((np.inf, -np.inf, 3e38, -2e38, 9e37)):
        som0[k::6, outside] = value
    if pixel:
        imgs[1, 0][pixel], imgs[3, 0][pixel] = -3e38, 2e38
    F = np.full((N, N), 1e-8, np.float32)
    F[:, 1::4] *= np.float32(-1.0)
    F[:, 2::7] = 0.0
    want = som0.reshape(N, -1).copy()
    want_bmu = O.train(O.shape(N, 1, I, D, nrot, True, ed, capi.QUADRATIC, ed_type), want, imgs, F)
    lost = np.isnan(want)
    assert lost.any() and np.isinf(want).any()
    with capi.Context(N, 1, I, D, nrot, True, ed, capi.QUADRATIC, ed_type, F) as ctx:
        ctx.set_som(som0.reshape(N, -1))
        bmu, som = ctx.train(imgs), ctx.get_som()
    assert np.array_equal(bmu, want_bmu) and np.array_equal(np.isnan(som), lost) and np.array_equal(bits(som)[~lost], bits(want)[~lost])


def test_resident_symmetric_trainer_tries_again(monkeypatch):
    """After a launch that gave up, the trainer takes the other form for some 256 images and is then resident again."""
    monkeypatch.setenv("PINK_HIP_RESIDENT_SPIN_LIMIT", "0")
    N, C_, I, D, nrot, ed, ed_type = 6, 2, 18, 12, 132, 8, capi.UINT8
    rng = np.random.default_rng(8)
    som0 = rng.random((N, C_ * D * D), dtype=np.float32)
    imgs = rng.random((320, C_, I, I), dtype=np.float32)
    F = capi.make_update_factors(capi.CARTESIAN, [N], capi.GAUSSIAN, 1.0, 0.5)
    want = som0.copy()
    obmu = O.train(O.shape(N, C_, I, D, nrot, True, ed, capi.QUADRATIC, ed_type), want, imgs, F)
    with capi.Context(N, C_, I, D, nrot, True, ed, capi.QUADRATIC, ed_type, F) as ctx:
        ctx.set_som(som0)
        # gives up; the other form, for as many images as the pause lasts; resident and gives up; the other form
        bmu = np.concatenate([ctx.train(imgs[a:b]) for a, b in ((0, 5), (5, 265), (265, 270), (270, 320))])
        som, counts = ctx.get_som(), ctx.update_counts()
    assert np.array_equal(bmu, obmu) and np.array_equal(bits(som), bits(want)) and np.array_equal(counts, np.bincount(obmu, minlength=N))


def test_resident_trainers_side_by_side():
    """Resident trainers whose blocks do not fit the device together, a thread each: their launches take turns."""
    import threading
    N, I, D, nrot, ed, n, ed_type = 200, 40, 32, 36, 32, 90, capi.UINT16          # (200 of 256 compute units, twice)
    F = capi.make_update_factors(capi.CARTESIAN, [N], capi.GAUSSIAN, 1.0, 0.5)
    work, got = [], {}
    for k in range(3):
        rng = np.random.default_rng(k)
        som0, imgs = rng.random((N, D * D), dtype=np.float32), rng.random((n, 1, I, I), dtype=np.float32)
        want = som0.copy()
        work.append((som0, imgs, want, O.train(O.shape(N, 1, I, D, nrot, True, ed, capi.QUADRATIC, ed_type), want, imgs, F)))

    def train(k):
        som0, imgs = work[k][:2]
        with capi.Context(N, 1, I, D, nrot, True, ed, capi.QUADRATIC, ed_type, F, max_batch=6) as ctx:
            ctx.set_som(som0)
            got[k] = (np.concatenate([ctx.train(imgs[i:i + 30]) for i in range(0, n, 30)]), ctx.get_som())

    threads = [threading.Thread(target=train, args=(k,)) for k in range(len(work))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k, (_, _, want, bmu) in enumerate(work):
        assert np.array_equal(got[k][0], bmu) and np.array_equal(bits(got[k][1]), bits(want)), k


def test_resident_float_trainers_side_by_side():
    """... and float32 ones, each waiting for its own first images."""
    import threading
    trainers, done = [FloatTrainer(200, 40, 32, 36, 32) for _ in range(3)], []

    def train(t):
        for _ in range(3):
            t.groups(t.images(40))
        done.append(t)

    threads = [threading.Thread(target=train, args=(t,)) for t in trainers]
    for thread in threads:
        thread.start()
    for thread in threads:
        thread.join()
    assert len(done) == len(trainers)
    for t in trainers:
        t.check()


def test_resident_symmetric_training_is_queued():
    """pink_hip_train_device returns while the device still trains (uint8, the command line's sizes for 64-pixel images)."""
    import time
    from test_zz_no_alloc import Hip
    N, I, D, ed, n = 100, 64, 91, 45, 3000
    F = capi.make_update_factors(capi.CARTESIAN, [10, 10], capi.GAUSSIAN, 1.1, 0.2)
    hip = Hip()
    imgs, bmu = hip.upload(np.random.default_rng(4).random((n, 1, I, I), dtype=np.float32)), hip.alloc(4 * n)
    with capi.Context(N, 1, I, D, 360, True, ed, capi.QUADRATIC, capi.UINT8, F) as ctx:
        ctx.set_som(np.zeros((N, D * D), np.float32))
        ctx.train_device(imgs, 100, bmu)
        ctx.synchronize()
        start = time.perf_counter()
        ctx.train_device(imgs, n, bmu)
        queued = time.perf_counter() - start
        ctx.synchronize()
        whole = time.perf_counter() - start
    hip.release()
    say("queued after", queued, "of", whole)
    assert queued < 0.5 * whole


ORBIT_TRAIN_SHAPES = [
    (3, 1, 70, 99, 48, True, 95, capi.QUADRATIC, capi.UINT8, 5),       # 12 base rotations; an odd neuron
    (5, 1, 60, 100, 180, False, 91, capi.QUADRATIC, capi.UINT16, 4),   # unlike symmetries, four columns per neuron
    (4, 2, 64, 90, 132, True, 70, capi.QUADRATIC, capi.UINT8, 3),      # two channels
    (1030, 1, 40, 36, 48, True, 33, capi.QUADRATIC, capi.UINT16, 3),   # more neurons than the resident form takes
    (2, 1, 190, 120, 60, True, 110, capi.CIRCULAR, capi.UINT16, 3),    # an image beyond the LDS
    (2, 1, 260, 200, 24, True, 190, capi.QUADRATIC, capi.UINT16, 2),   # ... and its window too
    (1030, 1, 1, 3, 8, True, 3, capi.QUADRATIC, capi.UINT8, 2),        # an image of a pixel
]


@pytest.mark.parametrize("N,C_,I,D,nrot,flip,ed,shape_,ed_type,n", ORBIT_TRAIN_SHAPES)
def test_trainer_with_weights_in_orbit_order(N, C_, I, D, nrot, flip, ed, shape_, ed_type, n):
    """Integer trainers too large for the resident form: the region's weights stay in the order of the operand over a call."""
    say("orbit trainer", N, C_, I, D, nrot, flip, ed, shape_, ed_type, n)
    rng = np.random.default_rng(N + I + nrot)
    som0, imgs = rng.random((N, C_ * D * D), dtype=np.float32), rng.random((n, C_, I, I), dtype=np.float32)
    F = capi.make_update_factors(capi.CARTESIAN, [N], capi.GAUSSIAN, 1.0, 0.5)
    F[F < 0.01] = 0.0
    s = O.shape(N, C_, I, D, nrot, flip, ed, shape_, ed_type)
    want = som0.copy()
    obmu = O.train(s, want, imgs, F)
    for max_batch in (0, 2):
        with capi.Context(N, C_, I, D, nrot, flip, ed, shape_, ed_type, F, max_batch=max_batch) as ctx:
            ctx.set_som(som0)
            bmu = np.concatenate([ctx.train(imgs[:1]), ctx.train(imgs[1:])])
            som, counts = ctx.get_som(), ctx.update_counts()
            d, ssd, best = ctx.distance(imgs[0])
        assert np.array_equal(bmu, obmu) and np.array_equal(bits(som), bits(want)), max_batch
        assert np.array_equal(counts, np.bincount(obmu, minlength=N)), max_batch
        heat, rot = O.map_images(s, want, imgs[:1])
        assert np.array_equal(best, rot[0]) and np.array_equal(bits(np.sqrt(d.astype(np.float64)).astype(np.float32)), bits(heat[0])), max_batch


SCREENED_TRAIN_SHAPES = [
    (1037, 1, 60, 44, 360, True, 37, capi.QUADRATIC, 3, "blobs"),      # a block of two neurons at the end
    (515, 2, 70, 60, 360, False, 53, capi.QUADRATIC, 3, "blobs"),      # four columns per neuron
    (700, 1, 80, 70, 264, True, 61, capi.CIRCULAR, 3, "noise"),        # 66 base rotations: two lists
    (640, 1, 90, 128, 128, True, 90, capi.QUADRATIC, 3, "zeros"),      # most variants alike: every variant of every neuron summed
    (523, 1, 70, 60, 452, True, 49, capi.QUADRATIC, 3, "grown"),       # some neurons keep all variants; 113 base rotations
    (517, 1, 70, 62, 360, True, 52, capi.QUADRATIC, 19, "flat"),      # ... image after image: no product for some of them, then again
    (1037, 1, 60, 44, 360, True, 37, capi.QUADRATIC, 3, "close"),      # 18000 variants listed
    (1037, 1, 60, 44, 360, True, 37, capi.QUADRATIC, 3, "closer"),     # 16300
    (1200, 1, 64, 50, 180, True, 50, capi.QUADRATIC, 3, "nan"),
    (1037, 1, 60, 44, 360, True, 37, capi.QUADRATIC, 3, "flux"),       # every variant close, squares of errors no float32
    (3100, 1, 40, 30, 360, True, 22, capi.QUADRATIC, 3, "steps"),      # sums that meet ties; runs of 8
    (900, 1, 60, 56, 360, True, 45, capi.QUADRATIC, 3, "steps"),       # ... of 32
    (1037, 1, 60, 44, 360, True, 37, capi.QUADRATIC, 5, "tail"),       # factors down to nothing: which neurons do they move?
    (1000, 1, 60, 44, 360, True, 43, capi.CIRCULAR, 5, "tail"),
    (9, 1, 100, 96, 360, True, 91, capi.QUADRATIC, 3, "blobs"),        # few neurons, long rows
    (49, 1, 180, 176, 128, True, 171, capi.QUADRATIC, 2, "noise"),     # ... longer than the LDS holds beside their operand
    (30, 2, 80, 80, 4, True, 73, capi.CIRCULAR, 3, "steps"),           # the symmetries only
    (100, 1, 64, 60, 100, False, 60, capi.QUADRATIC, 5, "tail"),
]


@pytest.mark.parametrize("N,C_,I,D,nrot,flip,ed,shape_,n,kind", SCREENED_TRAIN_SHAPES)
def test_float_trainer_with_screened_distances(monkeypatch, N, C_, I, D, nrot, flip, ed, shape_, n, kind):
    """Large float32 trainers sum the variants that a product of rounded values leaves: the oracle's bits, which sums them all."""
    monkeypatch.setenv("PINK_HIP_RESIDENT_TRAINER", "0")
    say("screened float trainer", N, C_, I, D, nrot, flip, ed, shape_, n, kind)
    F = capi.make_update_factors(capi.CARTESIAN, [N], capi.MEXICAN_HAT if kind == "grown" else capi.GAUSSIAN, 1.0, 0.5)
    rng = np.random.default_rng(N + I)
    som0, imgs = rng.random((N, C_ * D * D), dtype=np.float32), rng.random((n, C_, I, I), dtype=np.float32)
    if kind == "blobs":
        x = np.linspace(-1, 1, I, dtype=np.float32)
        imgs = imgs * 0.1 + np.exp(-8 * (x[:, None] - imgs[:, :, :1, :1]) ** 2 - 20 * x[None, :] ** 2).astype(np.float32)
    elif kind == "zeros":
        imgs[imgs < 0.999] = 0.0
    elif kind == "flat":
        imgs[:-1] = 0.25
    elif kind == "grown":
        som0[::9] *= 3000.0                                            # (far above the images: distances differ by less than they round)
    elif kind == "nan":
        imgs[1, 0, I // 2, I // 2] = np.nan
    elif kind.startswith("close"):
        imgs = _nearly_round(rng, n, C_, I, 1.0, 0.02 if kind == "close" else 0.03)
    elif kind == "steps":
        # few bits in every value: images alike under the symmetries but for a few pixels, neurons a multiple of 2^-10 beside them
        half = np.rint(imgs * 4) / 4
        imgs = half + half[:, :, ::-1] + half[:, :, :, ::-1] + half[:, :, ::-1, ::-1]
        imgs = (imgs + imgs.transpose(0, 1, 3, 2)).astype(np.float32)
        imgs[:, :, I // 3, I // 2] += np.float32(2.0 ** -9)
        m = (I - D) // 2
        som0 = (imgs[0, :, m:m + D, m:m + D].reshape(1, -1) + np.rint((som0 - 0.5) * 2048) / 1024).astype(np.float32)
    elif kind == "tail":
        F = capi.make_update_factors(capi.CARTESIAN, [N], capi.GAUSSIAN, 90.0, 0.5) ** np.float32(1.7)
        F[:, ::5] *= np.float32(1e-8)
        som0[1::4] += np.float32(0.5)                                  # (no small weights)
        som0[2::4, ::D] *= np.float32(1e-12)
        som0[3::4, 7] = 0.0
        imgs[3] -= np.float32(0.25)
    elif kind == "flux":
        imgs, som0 = _nearly_round(rng, n, C_, I, 5e-19), som0 * np.float32(5e-19)
    if kind != "tail":
        F[np.abs(F) < 0.01] = 0.0
    s = O.shape(N, C_, I, D, nrot, flip, ed, shape_, capi.FLOAT)
    want = som0.copy()
    want_bmu = O.train(s, want, imgs, F)
    want_d, want_best = O.map_images(s, want, imgs[:1])
    if kind == "nan":       # (no order among such distances: the kernel that sums every variant is the measure)
        with capi.Context(N, C_, I, D, nrot, flip, ed, shape_, capi.FLOAT, F, kernel_choice=capi.KERNEL_VALU) as ctx:
            ctx.set_som(som0)
            want_bmu = ctx.train(imgs)
            want = ctx.get_som()
            d, _, want_best = ctx.distance(imgs[0])
            want_d, want_best = np.sqrt(d.astype(np.float64)).astype(np.float32)[None], want_best[None]
    lost = np.isnan(want)
    for max_batch in (0, 2):
        with capi.Context(N, C_, I, D, nrot, flip, ed, shape_, capi.FLOAT, F, max_batch=max_batch) as ctx:
            ctx.set_som(som0)
            bmu = np.concatenate([ctx.train(imgs[:1]), ctx.train(imgs[1:])])
            som, counts = ctx.get_som(), ctx.update_counts()
            d, _, best = ctx.distance(imgs[0])
        assert lost.any() == (kind == "nan")
        assert np.array_equal(bmu, want_bmu) and np.array_equal(counts, np.bincount(want_bmu, minlength=N)), max_batch
        assert np.array_equal(np.isnan(som), lost) and np.array_equal(bits(som)[~lost], bits(want)[~lost]), max_batch
        d = np.sqrt(d.astype(np.float64)).astype(np.float32)
        known = ~np.isnan(want_d[0])
        assert np.array_equal(np.isnan(d), ~known) and np.array_equal(bits(d)[known], bits(want_d[0])[known]), max_batch
        assert np.array_equal(best[known], want_best[0][known]), max_batch


def test_screened_float_trainer_after_an_image_without_bounds(monkeypatch):
    """An image that holds a NaN and an infinity beside the region: the largest value is then no number, and the weight that the
    infinity made infinite is moved by the smallest factor."""
    monkeypatch.setenv("PINK_HIP_RESIDENT_TRAINER", "0")
    say("screened float trainer after an image without bounds")
    N, I, D, nrot, ed, n = 9, 100, 96, 360, 91, 17
    rng = np.random.default_rng(3)
    som0 = (0.1 + 0.5 * rng.random((N, D, D))).astype(np.float32)
    imgs = np.full((n, 1, I, I), 0.3, np.float32)
    imgs[:, 0, 2:98, 2:98] = som0[[0] + (n - 2) * [7] + [5]]           # (fifteen images are not screened behind the first)
    imgs[0, 0, 2, 2], imgs[0, 0, 97, 97] = np.inf, np.nan
    F = np.zeros((N, N), np.float32)
    F[0], F[5] = 0.5, 1e-12
    want = som0.reshape(N, -1).copy()
    want_bmu = O.train(O.shape(N, 1, I, D, nrot, True, ed, capi.QUADRATIC, capi.FLOAT), want, imgs, F)
    assert want_bmu.tolist() == [0] + (n - 2) * [7] + [5]
    lost = np.isnan(want)
    assert lost.reshape(N, D, D)[0, 0, 0]
    with capi.Context(N, 1, I, D, nrot, True, ed, capi.QUADRATIC, capi.FLOAT, F, max_batch=n) as ctx:
        ctx.set_som(som0.reshape(N, -1))
        bmu, som = ctx.train(imgs), ctx.get_som()
    assert np.array_equal(bmu, want_bmu) and np.array_equal(np.isnan(som), lost) and np.array_equal(bits(som)[~lost], bits(want)[~lost])


@pytest.mark.parametrize("N,ed_type", [(9, capi.FLOAT), (9, capi.UINT8), (530, capi.UINT8)])
def test_train_with_any_factor_matrix(N, ed_type):
    # the C interface takes any N x N matrix, not only the symmetric ones that a distance functor gives
    say("train, factor matrix", N, ed_type)
    C_, I, D, nrot, flip, ed, n = 1, 12, 8, 4, True, 6, 3
    rng = np.random.default_rng(N + ed_type)
    som0 = rng.random((N, C_ * D * D), dtype=np.float32)
    imgs = rng.random((n, C_, I, I), dtype=np.float32)
    F = rng.random((N, N), dtype=np.float32) * np.float32(0.5)
    F[rng.random((N, N)) < 0.3] = 0.0
    assert not np.array_equal(F, F.T)
    s = O.shape(N, C_, I, D, nrot, flip, ed, capi.QUADRATIC, ed_type)
    want = som0.copy()
    obmu = O.train(s, want, imgs, F)
    with capi.Context(N, C_, I, D, nrot, flip, ed, capi.QUADRATIC, ed_type, F) as ctx:
        ctx.set_som(som0)
        bmu = ctx.train(imgs)
        som = ctx.get_som()
    assert np.array_equal(bmu, obmu)
    assert np.array_equal(bits(som), bits(want))


def test_contexts_of_different_sizes_side_by_side():
    # LDS limits are set per kernel, not per context: a context created later with smaller images must
    # not take away what an earlier one needs (uint8 mappers of 150 and 100 pixels, trainers of 181 and 44)
    say("contexts side by side")
    rng = np.random.default_rng(77)
    made = []
    for (I, D, ed, et, F) in ((150, 30, 20, capi.UINT8, None), (100, 30, 20, capi.UINT8, None),
                              (128, 181, 90, capi.UINT16, capi.make_update_factors(capi.CARTESIAN, [4], capi.GAUSSIAN, 1.0, 0.5)),
                              (64, 44, 32, capi.UINT16, capi.make_update_factors(capi.CARTESIAN, [4], capi.GAUSSIAN, 1.0, 0.5))):
        ctx = capi.Context(4, 1, I, D, 8, True, ed, capi.QUADRATIC, et, F)
        som = rng.random((4, D * D), dtype=np.float32)
        img = rng.random((1, I, I), dtype=np.float32)
        ctx.set_som(som)
        made.append((ctx, som, img, I, D, ed, et))
    try:
        for ctx, som, img, I, D, ed, et in made:          # the first contexts run after the last was created
            s = O.shape(4, 1, I, D, 8, True, ed, capi.QUADRATIC, et)
            od, ossd, obest = O.distance_matrix(s, som, O.rotated_images(img, 1, I, D, 8, True))
            d, ssd, best = ctx.distance(img)
            assert np.array_equal(ssd, ossd) and np.array_equal(best, obest)
    finally:
        for m in made:
            m[0].close()


@pytest.mark.parametrize("ed_type,factor", [(capi.UINT8, 255), (capi.UINT16, 65535)])
def test_largest_matrix_core_region_with_extreme_data(ed_type, factor):
    # 65 025 region elements, all of them at one end of the range in both operands: the byte-plane dot
    # products are as large as they get (closed form: 0, and factor^2 * elements)
    say("largest region on the matrix cores", ed_type)
    D = 255
    som = np.zeros((2, D * D), np.float32)
    som[1] = 1.0
    with capi.Context(2, 1, D, D, 1, False, D, capi.QUADRATIC, ed_type) as ctx:
        assert ctx.distance_kernel == capi.KERNEL_MFMA_GEMM
        ctx.set_som(som)
        for value in (0.0, 1.0):
            d, ssd, best = ctx.distance(np.full((1, D, D), value, np.float32))
            want = [0, factor * factor * D * D] if value == 0.0 else [factor * factor * D * D, 0]
            assert ssd.tolist() == want and best.tolist() == [0, 0]


def test_reference_mapper_known_answers():
    # test/CudaTest/mapper.cu:115-119 in float, uint8 and uint16; circular_ed.cu:23-53
    for som_dim, nd, idim, ed, nrot, flip in [(1, 2, 2, 2, 1, False), (1, 3, 3, 2, 1, False), (1, 3, 3, 2, 360, False),
                                              (2, 3, 3, 2, 360, False), (2, 3, 3, 2, 360, True)]:
        N = som_dim * som_dim
        for ed_type in (capi.FLOAT, capi.UINT8, capi.UINT16):
            with capi.Context(N, 1, idim, nd, nrot, flip, ed, capi.QUADRATIC, ed_type) as ctx:
                ctx.set_som(np.ones((N, nd * nd), np.float32))
                heat, _ = ctx.map(np.zeros((idim, idim), np.float32))
            assert heat.ravel().tolist() == [2.0] * N
    image = np.zeros(16, np.float32)
    image[4] = 1.0
    som = np.zeros(64, np.float32)
    som[4], som[18], som[43], som[61] = 1.0, 0.5, 0.8, 0.3
    with capi.Context(4, 1, 4, 4, 4, False, 4, capi.CIRCULAR, capi.FLOAT) as ctx:
        ctx.set_som(som)
        heat, best = ctx.map(image)
    assert np.allclose(heat.ravel(), [0.0, 0.5, 0.2, 0.7], atol=0.01)
    assert best.ravel().tolist() == [0, 1, 2, 3]


def test_map_full_size_properties():
    """cfg 1 at a size the oracle does not cover: properties that hold at any size."""
    w = synthetic.WORKLOADS["cfg1"]
    n = 2000
    imgs = synthetic.images(w, n)
    som = synthetic.initial_som(w)
    with synthetic.make_context(w) as ctx:
        ctx.set_som(som)
        heat, best = ctx.map(imgs)
        heat2, best2 = ctx.map(imgs[::-1])
        # rotating an image by a quarter turn permutes its variants: same heatmap, shifted index
        turned = np.ascontiguousarray(np.rot90(imgs[:50], k=-1, axes=(2, 3)))
        heat3, best3 = ctx.map(turned)
    assert np.array_equal(bits(heat2[::-1]), bits(heat)) and np.array_equal(best2[::-1], best)   # order-independent
    assert (heat >= 0).all() and np.isfinite(heat).all() and (best < w.R).all()
    assert np.array_equal(bits(heat3), bits(heat[:50]))


def test_host_buffers_in_pieces_match_smaller_calls():
    """Inputs beyond 64 MB go to the device piece by piece while the kernels of the piece before run, a mapper's
    inputs from 32 MB on through two pinned buffers that several host threads fill side by side (147 MB here: pieces
    that are no multiple of the 8 MB buffers): the results are those of calls small enough to go in one plain copy
    (1500 images, 25 MB)."""
    w = synthetic.WORKLOADS["cfg1"]
    n = 9000                                                   # 147 MB of images: three pieces
    imgs = synthetic.images(w, n)
    say("pieces: map", n)
    with synthetic.make_context(w) as ctx:
        ctx.set_som(synthetic.initial_som(w))
        heat, best = ctx.map(imgs)
        parts = [ctx.map(imgs[i:i + 1500]) for i in range(0, n, 1500)]
    assert np.array_equal(bits(heat), bits(np.concatenate([p[0] for p in parts])))
    assert np.array_equal(best, np.concatenate([p[1] for p in parts]))
    w = synthetic.WORKLOADS["cfg3"]
    n = 1200                                                   # 144 MB of three-channel images: three pieces
    imgs = synthetic.images(w, n)
    tiny = dict(N=16, dims=[4, 4])
    F = capi.make_update_factors(capi.CARTESIAN, tiny["dims"], capi.GAUSSIAN, 1.1, 0.2)
    som0 = synthetic.mt19937_uniform(tiny["N"] * w.channels * 40 * 40, 7).reshape(tiny["N"], -1)
    say("pieces: train", n)
    results = []
    for step in (n, 200):
        with capi.Context(tiny["N"], w.channels, w.image_dim, 40, 8, True, 30, capi.QUADRATIC, capi.UINT8, F) as ctx:
            ctx.set_som(som0)
            bmu = np.concatenate([ctx.train(imgs[i:i + step]) for i in range(0, n, step)])
            results.append((bmu, ctx.get_som(), ctx.update_counts()))
    assert np.array_equal(results[0][0], results[1][0]) and np.array_equal(bits(results[0][1]), bits(results[1][1]))
    assert np.array_equal(results[0][2], np.bincount(results[0][0], minlength=tiny["N"]))


def test_large_transfers_of_several_threads_at_once():
    """Six threads, each with its own mapper or trainer and host buffers of some MB: four have pinned pieces, the others none."""
    import threading
    N, D, n = 36, 64, 700
    rng = np.random.default_rng(12)
    som = rng.random((300, D * D), dtype=np.float32)
    imgs = [rng.random((n, 1, D, D), dtype=np.float32) for _ in range(6)]
    start, bad = threading.Barrier(6), []

    def work(k):
        trainer = k % 3 == 2                              # (a trainer's large transfer is its SOM)
        size = 300 if trainer else N
        factors = capi.make_update_factors(capi.CARTESIAN, [size], capi.GAUSSIAN, 1.0, 0.3) if trainer else None
        with capi.Context(size, 1, D, D, 4, True, 20, capi.QUADRATIC, capi.UINT8, factors) as ctx:
            ctx.set_som(som[:size])
            if trainer:
                ctx.train(imgs[k][:20])
                want = ctx.get_som()
                start.wait()
                got = [ctx.get_som() for _ in range(20)]
                bad.extend(k for g in got if not np.array_equal(bits(g), bits(want)))
            else:
                pieces = [ctx.map(imgs[k][i:i + 50]) for i in range(0, n, 50)]        # (below 1 MB a piece)
                want = [np.concatenate(p) for p in zip(*pieces)]
                start.wait()
                for _ in range(8):
                    heat, best = ctx.map(imgs[k])
                    if not (np.array_equal(bits(heat), bits(want[0])) and np.array_equal(best, want[1])):
                        bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_empty_inputs_are_no_ops():
    w = synthetic.WORKLOADS["cfg4"]
    som = synthetic.initial_som(w)
    none = np.empty((0, w.channels, w.image_dim, w.image_dim), np.float32)
    with synthetic.make_context(w) as ctx:
        ctx.set_som(som)
        assert ctx.train(none).shape == (0,)
        assert np.array_equal(bits(ctx.get_som()), bits(som))
    with capi.Context(w.som_size, w.channels, w.image_dim, w.neuron_dim, w.num_rot, w.use_flip, w.ed_dim,
                      w.ed_shape, w.ed_type) as ctx:
        ctx.set_som(som)
        heat, best = ctx.map(none)
        assert heat.shape == (0, w.som_size) and best.shape == (0, w.som_size)


@pytest.mark.parametrize("ed_type", [capi.UINT8, capi.UINT16])
def test_out_of_range_pixels_saturate_like_the_oracle(ed_type):
    """Values outside [0, 1] (undefined in the reference) quantise to the ends of the range on every
    integer path, 1.0 exactly to the top value."""
    N, C_, I, D, nrot, flip, ed = 20, 1, 24, 18, 40, True, 16
    rng = np.random.default_rng(5)
    som = (rng.random((N, D * D), dtype=np.float32) * 2 - 0.5).astype(np.float32)
    imgs = (rng.random((6, C_, I, I), dtype=np.float32) * 2 - 0.5).astype(np.float32)
    imgs[0, 0, :4, :4] = 1.0
    som[0, :9] = [1.0, 0.0, -0.0, 2.0, -3.0, 1.0000001, 0.99999994, 0.5, 1e-9]
    s = O.shape(N, C_, I, D, nrot, flip, ed, O.QUADRATIC, ed_type)
    oheat, obest = O.map_images(s, som, imgs)
    for choice in (capi.KERNEL_AUTO, capi.KERNEL_VALU, capi.KERNEL_MFMA_GEMM):
        with capi.Context(N, C_, I, D, nrot, flip, ed, capi.QUADRATIC, ed_type, kernel_choice=choice) as ctx:
            ctx.set_som(som)
            heat, best = ctx.map(imgs)
        assert np.array_equal(bits(heat), bits(oheat)) and np.array_equal(best, obest), choice


def test_train_full_size_is_deterministic_and_counts_every_image():
    """cfg 4 at its full size (60 000 images), where the oracle is not run: two runs agree bit for
    bit, every image gets a best-matching neuron, and a second epoch moves the map less than the first."""
    w = synthetic.WORKLOADS["cfg4"]
    imgs = synthetic.images(w)
    som0 = synthetic.initial_som(w)
    runs = []
    for _ in range(2):
        with synthetic.make_context(w) as ctx:
            ctx.set_som(som0)
            bmu = ctx.train(imgs)
            som1 = ctx.get_som()
            ctx.train(imgs)
            som2 = ctx.get_som()
        runs.append((bmu, som1, som2))
    assert np.array_equal(runs[0][0], runs[1][0]) and np.array_equal(bits(runs[0][1]), bits(runs[1][1]))
    bmu, som1, som2 = runs[0]
    assert bmu.shape == (w.n_images,) and bmu.max() < w.som_size
    assert np.bincount(bmu, minlength=w.som_size).sum() == w.n_images
    assert np.isfinite(som2).all()
    assert np.abs(som2 - som1).mean() < np.abs(som1 - som0).mean()


def test_mfma_kernel_refused_where_it_does_not_apply():
    with pytest.raises(capi.PinkError):
        capi.Context(200, 1, 16, 12, 8, True, 8, capi.QUADRATIC, capi.UINT8, kernel_choice=capi.KERNEL_MFMA)
    with pytest.raises(capi.PinkError):
        capi.Context(16, 1, 16, 12, 8, True, 8, capi.QUADRATIC, capi.FLOAT, kernel_choice=capi.KERNEL_MFMA)


@pytest.mark.parametrize("name,choice,distance_launches,update_launches", [
    # a small float32 trainer: a distance launch applies the update of the image before it; the group ends with one
    # launch for the neurons' full images and the last image's update
    ("cfg0", capi.KERNEL_AUTO, 5, 2),
    ("cfg4", capi.KERNEL_MFMA_GEMM, 5, 5),
    ("cfg4", capi.KERNEL_AUTO, 0, 1),       # a small uint8 trainer: one resident launch for the group
])
def test_profiling_counts_launches(name, choice, distance_launches, update_launches):
    w = synthetic.WORKLOADS[name]
    with synthetic.make_context(w, kernel_choice=choice) as ctx:
        ctx.set_som(synthetic.initial_som(w))
        ctx.set_profiling(True)
        ctx.train(synthetic.images(w, 5))
        t = ctx.kernel_times()
        ctx.set_profiling(False)
    # variants are prepared for a group of images per launch; distance and update run per image
    assert t["rotate"][0] == 1 and t["distance"][0] == distance_launches and t["update"][0] == update_launches
    assert all(ms >= 0 for _, ms in t.values())
