"""GPU: what the entry points promise beside their values: which work a read waits for, what a call's scratch may
hold, that a call gives the same twice, inputs at the end of the ranges that they take."""
import ctypes
import threading

import numpy as np
import pytest
import torch

from libfusion_amd import capi
from tests.helpers import triangles_in_hash_order

pytestmark = pytest.mark.gpu

FP32, MIXED = capi.PRECISION_FP32, capi.PRECISION_MIXED


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def room_images(K, n, seed):
    """n frames of patches at several depths around the origin, as images with poses (device pose24)."""
    rng = np.random.default_rng(seed)
    imgs, poses = [], []
    for _ in range(n):
        patches = rng.choice([0, 700, 900, 1300, 2100], (K.height // 8 + 1, K.width // 8 + 1))
        d16 = np.kron(patches, np.ones((8, 8), int))[:K.height, :K.width] + rng.integers(0, 4, (K.height, K.width))
        img = capi.Image(K, 1)
        img.upload(dev(d16.astype(np.uint16)), dev(rng.integers(0, 256, (K.height, K.width, 3)).astype(np.uint8)), 1e-3)
        imgs.append(img)
        T = np.eye(4)
        a = rng.uniform(-0.3, 0.3)
        T[:3, :3] = [[np.cos(a), 0, np.sin(a)], [0, 1, 0], [-np.sin(a), 0, np.cos(a)]]
        T[:3, 3] = rng.uniform(-0.2, 0.2, 3)
        poses.append(T)
    return imgs, poses


def by_block(m):
    """A map's sdf codes, weights (words of a mixed map) and colours by block coordinate."""
    n = int(m.counters()[capi.CNT_ALLOCATED])
    b = m.blocks()
    order = np.lexsort(b.T)
    rgb = m.t["rgb"][: 1536 * n].view(n, -1).cpu().numpy()[order] if m.params.precision == FP32 else None
    return [b[order], m.t["sdf"][: 512 * n].view(n, 512).cpu().numpy()[order],
            m.t["weight"][: 512 * n].view(n, 512).cpu().numpy()[order]] + ([rgb] if rgb is not None else [])


@pytest.mark.parametrize("n", [1, 12])
def test_mixed_refusion_gives_the_same_twice(n):
    """A mixed re-fusion counts 2 n passes, whatever the order of its walks, and so rounds the weights (by their
    stochastic rounding, seeded by the count) the same in two runs from one map."""
    K = capi.intrinsics(96, 64, 80.0, 80.0, 47.5, 31.5)
    p = capi.map_params(1 << 16, 1 << 15, 0.01, 0.03, precision=MIXED)
    imgs, poses = room_images(K, n, 5)
    old = [dev(capi.pose24(T)) for T in poses]
    new = []
    for T in poses:
        T[:3, 3] += 0.015
        new.append(dev(capi.pose24(T)))
    base = capi.Map(p, K.width, K.height)
    for img, T in zip(imgs, old):
        base.update_image(img, T)
    before = int(base.counters()[capi.CNT_FUSE_PASSES])
    assert before == n
    runs = []
    for _ in range(4):
        m = capi.Map(p, K.width, K.height)
        base.copy_to(m)
        m.refuse_keyframes(imgs, old, new)
        torch.cuda.synchronize()
        assert int(m.counters()[capi.CNT_FUSE_PASSES]) == before + 2 * n
        runs.append(by_block(m))
    for r in runs[1:]:
        assert all(np.array_equal(x, y) for x, y in zip(r, runs[0]))
    for img in imgs:
        img.close()


# at the origin; tens of kilometres from it, where a float coordinate is good to a fifth or to half a voxel; a camera
# whose unit is a quarter of the map's, and four of them
@pytest.mark.parametrize("offset,unit", [((0, 0, 0), 1.0), ((30000, -9000, 17000), 1.0), ((-61000, 0, 3000), 1.0),
                                         ((0, 0, 0), 0.25), ((100, 50, -20), 4.0)])
def test_refusion_at_any_pose(offset, unit):
    """Re-fusion leaves the voxels seen, and their weights, that de-integrating and fusing one keyframe after the
    other does (the same float arithmetic per voxel), wherever the cameras are and whatever their unit."""
    K = capi.intrinsics(160, 96, 130.0, 130.0, 79.5, 47.5)
    voxel = 0.01 * max(unit, 0.5)
    p = capi.map_params(1 << 17, 1 << 16, voxel, 3 * voxel)
    imgs, poses = room_images(K, 5, 9)

    def pose24(T):  # T_wc = unit R, t and its inverse
        R, t = T[:3, :3], T[:3, 3] * unit + np.asarray(offset, float)
        wc = np.concatenate([unit * R, t[:, None]], 1)
        cw = np.concatenate([R.T / unit, -(R.T @ t / unit)[:, None]], 1)
        return dev(np.concatenate([wc.ravel(), cw.ravel()]).astype(np.float32))

    old = [pose24(T) for T in poses]
    new = []
    for k, T in enumerate(poses):
        T[:3, 3] += (0.02, -0.01, 0.013 * (k - 2))
        new.append(pose24(T))
    base, seq, one = (capi.Map(p, K.width, K.height) for _ in range(3))
    for img, T in zip(imgs, old):
        base.update_image(img, T)
    base.copy_to(seq)
    base.copy_to(one)
    one.refuse_keyframes(imgs, old, new)
    for img, T in zip(imgs, old):
        seq.deintegrate_image(img, T)
    for img, T in zip(imgs, new):
        seq.update_image(img, T)
    torch.cuda.synchronize()
    (bo, _, wo, _), (bs, _, ws, _) = by_block(one), by_block(seq)
    assert int(seq.counters()[capi.CNT_OVERFLOW]) == 0 and (ws > 0).sum() > 5000
    assert np.array_equal(bo, bs)
    assert np.array_equal(wo, ws), int((wo != ws).sum())
    for img in imgs:
        img.close()


# a single workgroup, 45 of them, the capped grid
@pytest.mark.parametrize("width,height", [(20, 15), (160, 144), (640, 480)])
def test_reduction_sums_inside_the_scratch(width, height):
    """sum29 anywhere in the scratch: the rows, the flags, its middle, its end.  The same sums as beside it."""
    rng = np.random.default_rng(4)
    K = capi.intrinsics(width, height, 1.2 * width, 1.2 * width, (width - 1) / 2, (height - 1) / 2)
    d = (1.0 + 0.1 * rng.random((height, width))).astype(np.float32)
    x, y = np.meshgrid(np.arange(width), np.arange(height))
    v = np.stack([d * (x - K.cx) / K.fx, d * (y - K.cy) / K.fy, d, np.ones_like(d)], -1).astype(np.float32)
    n = rng.normal(size=(height, width, 4)).astype(np.float32)
    n[..., :3] /= np.linalg.norm(n[..., :3], axis=-1, keepdims=True)
    I, g = (rng.random((height, width)).astype(np.float32) * s for s in (200, 20))
    t = [dev(a) for a in (v, n, v + np.float32(0.001), n, I, I + 1, g, g)]
    lib, P, pose = capi.load(), capi.ptr, dev(np.eye(4, dtype=np.float32)[:3].ravel())
    size = lib.lf_reduce_scratch_floats()
    scratch = torch.zeros(size + 64, device="cuda")

    def both(at):
        out = []
        st = capi.stream_ptr()
        s = scratch[at: at + 29]
        for _ in range(3):
            capi.check(lib.lf_icp_reduce(P(t[0]), P(t[1]), P(t[2]), P(t[3]), width, height, P(pose), ctypes.byref(K),
                                         P(scratch), P(s), st))
            out.append(s.cpu().numpy().copy())
            capi.check(lib.lf_rgb_step(P(t[4]), P(t[5]), P(t[2]), P(t[6]), P(t[7]), width, height, 5.0, P(pose),
                                       ctypes.byref(K), P(scratch), P(s), st))
            out.append(s.cpu().numpy().copy())
        return out

    want = both(size)  # behind the scratch
    assert want[0][28] > 100 and want[1][28] > 100
    for at in (0, 1, 512 * 14, 512 * 29 - 15, 512 * 29 + 3, 512 * 31 - 29, 512 * 31, 512 * 31 + 17, size // 2, size - 29):
        assert all(np.array_equal(a, b) for a, b in zip(both(at), want)), at


@pytest.mark.parametrize("precision", [FP32, MIXED])
def test_mesh_of_an_sdf_plane_between_other_data(precision):
    """A caller's sdf plane that starts on no 4-byte boundary: the same triangles as from one that does."""
    from tests.test_gpu_kernels import map_of_blocks
    rng = np.random.default_rng(8)
    pos = np.array([(x, y, z) for x in range(3) for y in range(2) for z in range(2)])
    value = rng.choice([-1.0, 1.0], (len(pos), 512))
    sdf = (value.astype(np.float16).view(np.int16) if precision == MIXED else (value * 32767).astype(np.int16))
    weight = np.full((len(pos), 512), 0x70, np.uint8) if precision == MIXED else np.ones((len(pos), 512), np.float32)
    m = map_of_blocks(precision, pos, sdf, weight, rng.integers(0, 256, (len(pos), 3, 512)).astype(np.uint8))
    want, _, n = m.mesh(0, 100000)
    aside = torch.zeros(m.t["sdf"].numel() + 8, dtype=torch.int16, device="cuda")
    for at in (1, 3, 5):
        plane = aside[at: at + m.t["sdf"].numel()]
        plane.copy_(m.t["sdf"])
        m.storage.sdf = plane.data_ptr()
        got, _, k = m.mesh(0, 100000)
        assert k == n > 1000
        assert np.array_equal(*(triangles_in_hash_order(t.cpu().numpy()) for t in (got, want)))


# inside the block directory, across its upper and its lower end, beside it, far outside it
@pytest.mark.parametrize("centre", [(0, 0, 3), (126, 1, 4), (-127, -126, 2), (2, 0, 127), (3, 131, 2), (-200, 150, 260)])
def test_mixed_raycast_around_the_directory(centre):
    """A mixed map's raycast of a rough surface with holes, vertex for vertex and colour for colour that of an FP32 map
    of the same values: sdfs of -1 and 1, which both storages hold exactly."""
    from tests.test_gpu_kernels import map_of_blocks
    rng = np.random.default_rng(31)
    width, height, voxel = 72, 48, 0.01
    pos = np.array([(x, y, z) for x in range(-4, 4) for y in range(-4, 4) for z in range(-1, 2)]) + centre
    pos = pos[rng.random(len(pos)) < 0.85]
    z, y, x = np.meshgrid(*[np.arange(8)] * 3, indexing="ij")
    at = pos[:, :, None] * 8 + np.stack([x.ravel(), y.ravel(), z.ravel()])[None]
    surface = centre[2] * 8 + 4 + 3 * np.sin(0.3 * at[:, 0]) * np.cos(0.2 * at[:, 1]) + rng.random((len(pos), 512))
    inside = at[:, 2] > surface
    seen = rng.random((len(pos), 512)) < 0.93
    rgb = rng.integers(0, 256, (len(pos), 3, 512)).astype(np.uint8)
    one, minus = np.float16(1).view(np.int16), np.float16(-1).view(np.int16)
    codes = {FP32: np.where(seen, np.where(inside, -32767, 32767), capi.SDF_UNSEEN).astype(np.int16),
             MIXED: np.where(seen, np.where(inside, minus, one), -1).astype(np.int16)}
    weight = {FP32: seen.astype(np.float32), MIXED: (0x70 * seen).astype(np.uint8)}
    K = capi.intrinsics(width, height, 60.0, 60.0, (width - 1) / 2, (height - 1) / 2)
    for turn in (0.0, 0.4, -0.7):
        T = np.eye(4)
        T[:3, :3] = [[np.cos(turn), 0, np.sin(turn)], [0, 1, 0], [-np.sin(turn), 0, np.cos(turn)]]
        T[:3, 3] = (np.array(centre) + 0.5) * 0.08 - 0.7 * T[:3, 2]
        got = []
        for precision in (FP32, MIXED):
            m = map_of_blocks(precision, pos, codes[precision], weight[precision], rgb, voxel, size=(width, height))
            vm = torch.zeros((height, width, 4), device="cuda")
            col = torch.zeros((height, width, 3), dtype=torch.uint8, device="cuda")
            m.raycast_check_visibility(vm, dev(capi.pose24(T)), K, rgb_out=col)
            torch.cuda.synchronize()
            got.append((vm.cpu().numpy(), col.cpu().numpy()))
        hit = ~np.isnan(got[0][0][..., 0])
        assert hit.mean() > 0.2
        assert np.array_equal(got[0][0][hit], got[1][0][hit]) and np.isnan(got[1][0][~hit]).all()
        assert np.array_equal(got[0][1], got[1][1])


# a normal whose z is NaN, and a depth of 0 accepted by the range: frame weights of NaN and of infinity
@pytest.mark.parametrize("depth,normal", [(0.04, float("nan")), (0.0, 1.0)])
def test_mixed_colours_of_frames_without_a_finite_weight(depth, normal):
    """The means of such a frame's colours are NaN: they are stored as 255, as ever, the weight as 255 too."""
    w, h = 48, 32
    K = capi.intrinsics(w, h, 30.0, 30.0, (w - 1) / 2, (h - 1) / 2)
    p = capi.map_params(1 << 12, 1 << 12, 0.01, 0.05, precision=MIXED)
    p.zmin_update = 0.0
    m = capi.Map(p, w, h)
    pose = dev(capi.pose24(np.eye(4)))

    def fuse(d, nz, c):
        nmap = np.zeros((h, w, 4), np.float32)
        nmap[..., 2] = nz
        m.update_weighted(dev(np.full((h, w), d, np.float32)), dev(nmap), dev(np.full((h, w, 3), c, np.uint8)), pose, K)
        torch.cuda.synchronize()

    fuse(0.04, 0.5, 90)
    n = int(m.counters()[capi.CNT_ALLOCATED])
    words = m.t["weight"][: 512 * n].cpu().numpy().view(np.uint32)
    seen = (words & 0xFF) > 0
    assert seen.sum() > 200 and (words[seen] >> 8 == 0x5A5A5A).all()
    fuse(depth, normal, 30)
    after = m.t["weight"][: 512 * n].cpu().numpy().view(np.uint32)
    changed = seen & (after != words)
    assert changed.sum() > 50
    assert (after[changed] >> 8 == 0xFFFFFF).all()
    top = capi.load().lf_weight_code_dither(255.0, 0)
    assert (after[changed] & 0xFF >= top).all()


def batch_of(n, precision, graphs):
    """A batch of n 640x480 cameras of one moving scene each, and six frames of them."""
    from libfusion_amd.synth import Scene
    scenes = [Scene(1, 40 + k) for k in range(n)]
    K = [capi.intrinsics(640, 480, s.fx, s.fy, s.cx, s.cy) for s in scenes]
    p = capi.map_params(1 << 18, 1 << 15, 0.01, 0.03, precision=precision)
    b = capi.Batch([capi.system_config(k, p, 3, (10, 5, 3), s.depth_scale) for k, s in zip(K, scenes)])
    b.set_graphs(graphs)
    frames = []
    for f in range(6):
        pairs = [s.frame(f) for s in scenes]
        frames.append(([dev(d.view(np.int16)) for d, _ in pairs], [dev(c) for _, c in pairs]))
    torch.cuda.synchronize()
    return b, frames


@pytest.mark.parametrize("precision,graphs", [(FP32, False), (MIXED, True)])
def test_batch_reads_wait_for_the_steps_processed(precision, graphs):
    """A batch's pose, tracking result and counters right after the last step is enqueued are those after a
    synchronisation, every frame having moved the camera."""
    b, frames = batch_of(4, precision, graphs)
    before = None
    for upto in (2, 6):  # one read after the first frames, one with steps of a steady state behind it
        for d, c in frames[0 if upto == 2 else 2:upto]:
            b.process(d, c)
        pose = [b.pose(i, wait=True) for i in range(4)]
        b.synchronize()
        assert all(np.array_equal(p, b.pose(i)) for i, p in enumerate(pose))
        if before is not None:
            assert all(np.abs(p - q).max() > 1e-3 for p, q in zip(pose, before))
        before = pose
    # the other two reads, each the first after a step
    for read in (b.tracking, b.counters):
        b.process(*frames[5])
        now = [read(i) for i in range(4)]
        b.synchronize()
        assert all(np.array_equal(x, read(i), equal_nan=True) for i, x in enumerate(now))
    b.close()


@pytest.mark.parametrize("wait", [False, True])
def test_batch_poses_read_beside_the_steps(wait):
    """Poses read by another thread while the steps are enqueued are each the pose after one of the steps, in order,
    and after a synchronisation the last one's."""
    b, frames = batch_of(2, FP32, False)
    known = [b.pose(0)]
    assert np.array_equal(b.pose(0, wait=True), known[0])
    for d, c in frames:
        b.process(d, c)
        b.synchronize()
        known.append(b.pose(0))
    b.close()
    b, frames = batch_of(2, FP32, False)
    seen, done = [], threading.Event()

    def poll():
        while not done.is_set():
            seen.append(b.pose(0, wait=wait))

    t = threading.Thread(target=poll)
    t.start()
    for d, c in frames:
        b.process(d, c)
    done.set()
    t.join()
    b.synchronize()
    seen.append(b.pose(0))
    b.close()
    # the same frames through the same kernels: a step's pose differs by 1e-7 at most, a frame's motion is over 1e-3
    at = [int(np.argmin([np.abs(p - k).max() for k in known])) for p in seen]
    assert max(np.abs(p - known[i]).max() for p, i in zip(seen, at)) < 3e-7
    assert at == sorted(at) and at[-1] == len(known) - 1
