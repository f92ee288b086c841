"""GPU: what the entry points promise beside their values: which work a read waits for, what a call's scratch may
hold, that a call gives the same twice, inputs at the end of the ranges that they take."""
import threading

import numpy as np
import pytest
import torch

from libfusion_amd import capi

pytestmark = pytest.mark.gpu

FP32, MIXED = capi.PRECISION_FP32, capi.PRECISION_MIXED


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


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
