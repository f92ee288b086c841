"""GPU: kernels at the sizes where their tiling can go wrong, against plain numpy / torch restatements."""
import ctypes

import numpy as np
import pytest
import torch

from libfusion_amd import capi
from tests.helpers import triangles_in_hash_order

pytestmark = pytest.mark.gpu

FP32, MIXED = capi.PRECISION_FP32, capi.PRECISION_MIXED


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def map_of_blocks(precision, pos, sdf, weight, rgb, voxel_size=0.005, buckets=1 << 12, size=(64, 64)):
    """A map that holds the given blocks: pos int[n,3], sdf codes int16[n,512] (FP16 bits of a mixed map),
    weight float32[n,512] or weight codes uint8 of a mixed map, rgb uint8[n,3,512]."""
    n = len(pos)
    p = capi.map_params(buckets, n + 5, voxel_size, 3 * voxel_size, precision=precision)
    m = capi.Map(p, *size)
    lib = capi.load()
    keys = np.full(p.num_entries, -1, np.int64)
    slot_block = np.full(p.num_entries, -1, np.int32)
    block_pos = np.zeros((p.num_blocks, 4), np.int32)
    cells, occ = [], np.zeros(capi.OCC_WORDS, np.uint32)
    for b, (x, y, z) in enumerate(pos.tolist()):
        slot = lib.lf_compute_hash(x, y, z, p.num_buckets)
        while keys[slot] != -1:
            slot = (slot + 1) % p.num_entries
        keys[slot] = ((x & 0x1FFFFF) << 42) | ((y & 0x1FFFFF) << 21) | (z & 0x1FFFFF)
        slot_block[slot] = b
        block_pos[b] = (x, y, z, slot)
        o = lib.lf_occupancy_bit(x, y, z)
        occ[o >> 5] |= np.uint32(1 << (o & 31))
        if lib.lf_dir_cell(x, y, z) >= 0:
            cells.append((lib.lf_dir_cell(x, y, z), b))
    m.t["keys"].copy_(dev(keys))
    m.t["slot_block"].copy_(dev(slot_block))
    m.t["block_pos"].copy_(dev(block_pos.reshape(-1)))
    m.t["occupancy"].copy_(dev(occ.view(np.int32)))
    if cells:
        at, b = np.array(cells).T
        m.t["block_dir"][dev(at)] = dev(b.astype(np.int32))
    m.t["counters"][capi.CNT_ALLOCATED] = n
    m.t["sdf"][: n * 512] = dev(sdf.reshape(-1))
    if precision == MIXED:
        w = weight.astype(np.uint32)
        for k in range(3):
            w |= rgb[:, k].astype(np.uint32) << (8 + 8 * k)
        m.t["weight"][: n * 512] = dev(w.view(np.int32).reshape(-1))
    else:
        m.t["weight"][: n * 512] = dev(weight.reshape(-1))
        m.t["rgb"][: n * 1536] = dev(rgb.reshape(-1))
    return m


def mesh_of_blocks(pos, val, ok, rgb, vs):
    """Marching cubes of the blocks in float32 numpy: val float32[n,512], ok bool[n,512], rgb uint8[n,3,512]
    -> (vertices[t,9], normals[t,9], colours[t,9])."""
    edge, tri = capi.mc_tables()
    where = {tuple(q): b for b, q in enumerate(pos.tolist())}
    corner = np.array([(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)])
    ends = [(0, 1), (1, 2), (2, 3), (3, 0), (4, 5), (5, 6), (6, 7), (7, 4), (0, 4), (1, 5), (2, 6), (3, 7)]
    one = np.float32(1)
    out = []
    for b, q in enumerate(pos.tolist()):
        V, G, C = np.zeros((9, 9, 9), np.float32), np.zeros((9, 9, 9), bool), np.zeros((9, 9, 9, 3), np.uint8)  # z y x
        for k in range(8):
            d = (k & 1, k >> 1 & 1, k >> 2)
            nb = where.get((q[0] + d[0], q[1] + d[1], q[2] + d[2]))
            if nb is None:
                continue
            at = tuple(slice(8, 9) if e else slice(0, 8) for e in d[::-1])
            src = tuple(slice(0, 1) if e else slice(0, 8) for e in d[::-1])
            V[at] = val[nb].reshape(8, 8, 8)[src]
            G[at] = ok[nb].reshape(8, 8, 8)[src]
            C[at] = np.moveaxis(rgb[nb].reshape(3, 8, 8, 8), 0, -1)[src]
        z, y, x = np.meshgrid(*[np.arange(8)] * 3, indexing="ij")
        s = np.stack([V[z + c[2], y + c[1], x + c[0]] for c in corner], -1)
        g = np.all([G[z + c[2], y + c[1], x + c[0]] for c in corner], 0)
        ci = ((s < 0) << np.arange(8)).sum(-1) * g
        for iz, iy, ix in np.argwhere(edge[ci] != 0):
            c, sv = ci[iz, iy, ix], s[iz, iy, ix]
            base = np.float32([q[0] * 8 + ix, q[1] * 8 + iy, q[2] * 8 + iz])
            for t in range(0, 15, 3):
                if tri[c, t] < 0:
                    break
                vtx, col = [], []
                for e in tri[c, t:t + 3]:
                    i, j = ends[e]
                    a, d = sv[i], sv[j]
                    f = (np.float32(0) if abs(float(a)) < 1e-6 else one if abs(float(d)) < 1e-6 else
                         np.float32(0) if abs(float(a - d)) < 1e-6 else (np.float32(0) - a) / (d - a))
                    off = corner[i].astype(np.float32)
                    ax = int(np.flatnonzero(corner[i] != corner[j])[0])
                    off[ax] = one - f if corner[i][ax] else f
                    vtx.append((base + off) * np.float32(vs))
                    k = corner[i]
                    col.append(C[iz + k[2], iy + k[1], ix + k[0]])
                u, w = vtx[1] - vtx[0], vtx[2] - vtx[0]
                n = np.float32([u[1] * w[2] - u[2] * w[1], u[2] * w[0] - u[0] * w[2], u[0] * w[1] - u[1] * w[0]])
                with np.errstate(invalid="ignore", divide="ignore"):
                    n = n / np.sqrt((n[0] * n[0] + n[1] * n[1]) + n[2] * n[2])
                out.append((np.concatenate(vtx), np.tile(n, 3), np.concatenate(col)))
    v, n, c = (np.array(a) for a in zip(*out)) if out else (np.zeros((0, 9), np.float32),) * 3
    return v, n, c


# one block, a full row of neighbours, blocks on both sides of the block directory's end, a count that fills no
# workgroup; dense random signs (up to 5 triangles a cube, layers that overflow the triangle list) and sparse ones
@pytest.mark.parametrize("precision", [FP32, MIXED])
@pytest.mark.parametrize("shape,origin,dense", [((1, 1, 1), (0, 0, 0), 1.0), ((3, 2, 2), (-1, -1, 3), 0.85),
                                                ((2, 2, 2), (126, -129, 0), 0.5), ((3, 3, 1), (5, 0, -2), 0.02)])
def test_mesh_of_random_blocks(precision, shape, origin, dense):
    rng = np.random.default_rng(3)
    pos = np.array([(x + origin[0], y + origin[1], z + origin[2]) for z in range(shape[2]) for y in range(shape[1])
                    for x in range(shape[0])])
    n = len(pos)
    v = rng.uniform(-1, 1, (n, 512)) if dense > 0.1 else np.where(rng.random((n, 512)) < dense, -0.3, 0.7)
    v[rng.random((n, 512)) < 0.02] = 0.0
    seen = rng.random((n, 512)) < (dense if dense > 0.1 else 1.0)
    if precision == MIXED:
        codes = np.where(seen, v.astype(np.float16).view(np.int16), np.int16(-1)).astype(np.int16)
        val = codes.view(np.float16).astype(np.float32)
        weight = np.where(seen, rng.integers(1, 240, (n, 512)), 0).astype(np.uint8)
        w = capi.weight_values()[weight]
    else:
        codes = np.where(seen, (v * 32767).astype(np.int16), np.int16(-32768)).astype(np.int16)
        val = codes.astype(np.float32) / np.float32(32767)
        weight = w = np.where(seen, rng.choice([5e-4, 0.1, 7.0], (n, 512)), 0).astype(np.float32)
    rgb = rng.integers(0, 256, (n, 3, 512)).astype(np.uint8)
    m = map_of_blocks(precision, pos, codes, weight, rgb)
    vs = m.params.voxel_size
    for mode in (0, 1, 2):
        ok = w > 1e-3 if mode == 2 else w != 0
        ov, on, oc = mesh_of_blocks(pos, np.where(ok, val, 0).astype(np.float32), ok, rgb, vs)
        gv, gx, count = m.mesh(mode=mode, max_triangles=len(ov) + 64)
        assert count == len(ov) and len(gv) == len(ov)
        gv = gv.cpu().numpy().reshape(-1, 9)
        if mode == 0:
            assert np.array_equal(triangles_in_hash_order(gv.reshape(-1, 3, 3)), triangles_in_hash_order(ov.reshape(-1, 3, 3)))
            continue
        gx, ox = gx.cpu().numpy().reshape(-1, 9), on if mode == 1 else oc
        # rows ordered by vertices, then by the normal / colour (equal triangles of neighbouring cubes)
        rows = [np.concatenate([a, np.nan_to_num(b.astype(np.float32))], 1) + np.float32(0) for a, b in ((gv, gx), (ov, ox))]
        g, o = (r[np.lexsort(r.T[::-1])] for r in rows)
        assert np.array_equal(g[:, :9], o[:, :9])
        # normals: one rounding apart per operation of the cross product and the normalisation
        assert np.array_equal(g[:, 9:], o[:, 9:]) if mode == 2 else np.allclose(g[:, 9:], o[:, 9:], atol=1e-6)
    # a capacity inside the output: the count goes on, nothing is written beyond it
    cap = max(1, len(ov) - 70)
    out = torch.full((len(ov) + 64, 9), 7.0, device="cuda")
    got = ctypes.c_uint(0)
    rc = capi.load().lf_create_mesh(ctypes.byref(m.params), ctypes.byref(m.storage), capi.ptr(out), None, None, cap,
                                    ctypes.byref(got), capi.stream_ptr())
    full = int(m.counters()[capi.CNT_TRIANGLES])
    assert got.value == min(cap, full) and rc == (capi.LF_ERR_CAPACITY if full > cap else capi.LF_OK)
    assert torch.all(out[got.value:] == 7.0) and not torch.any((out[: got.value] == 7.0).all(1))


def frame_pair(K, width, height):
    """Two neighbouring views of the orbit scene: (reference vmap, rgb), (source vmap, rgb) on the device."""
    from libfusion_amd.synth import Scene
    sc = Scene(1, 7)
    out = []
    for i in (0, 1):
        d, c = sc.render(sc.pose(i), width, height, K.fx, K.fy, K.cx, K.cy, frame_id=i)
        z = d.astype(np.float32) * np.float32(sc.depth_scale)
        u, v = np.meshgrid(np.arange(width, dtype=np.float32), np.arange(height, dtype=np.float32))
        m = np.stack([z * (u - K.cx) / K.fx, z * (v - K.cy) / K.fy, z, np.ones_like(z)], -1)
        m[~((z > 0.3) & (z < 5))] = (np.nan, np.nan, np.nan, -1)
        out.append((dev(m), dev(c)))
    return out


# one workgroup, 66 partial rows (more than a wavefront's lanes), 263 pixel blocks on the 256 workgroups of a lone
# tracker; the last with a coarser level below it
@pytest.mark.parametrize("width,height,levels", [(24, 16, 1), (192, 176, 1), (400, 336, 1), (400, 336, 2)])
def test_gauss_newton_steps_chain(width, height, levels):
    """A schedule run at once is its steps run one call at a time, each started where the one before ended: the
    solve that a launch finds at its head is the previous step's.  One step a level: a level's later steps take
    the residual deviation of the step before them, which a call starts without."""
    f = 525.0 * width / 640
    K = capi.intrinsics(width, height, f, f, (width - 1) / 2, (height - 1) / 2)
    ref, src = frame_pair(K, width, height)
    t = capi.Tracker(K, levels)
    for name, (v, c) in (("reference", ref), ("source", src)):
        t.set("set_%s_vmap" % name, v)
        t.set("set_%s_image" % name, c)
    _, _, whole = t.compute_transform((1,) * levels, np.eye(4))
    sums, est = t.sums(), np.eye(4)
    for level in range(levels - 1, -1, -1):
        _, _, upd = t.compute_transform(tuple(int(k == level) for k in range(levels)), est)
        est = np.linalg.inv(upd)
    # FP64 but for the pose that the rows are taken at, which an inversion may round to its other float
    assert np.allclose(np.linalg.inv(est), whole, rtol=0, atol=1e-6)
    assert np.allclose(t.sums(), sums, rtol=1e-3, atol=1e-5 * np.abs(sums[:27]).max())
    if levels > 1:
        return
    # against the stand-alone reduction on the same maps and pose, which adds the same float32 rows up in
    # float32: every correspondence counted, and r^2 within the rounding of a sum of at most 2^18 terms
    lib = capi.load()

    def plane(source, which):
        out = ctypes.c_void_p()
        capi.check(lib.lf_tracker_plane(t.h, source, 0, which, ctypes.byref(out)))
        return out
    pose = dev(np.eye(4, dtype=np.float32)[:3])
    scratch, out = torch.empty(lib.lf_reduce_scratch_floats(), device="cuda"), torch.empty(29, device="cuda")
    capi.check(lib.lf_icp_reduce(plane(1, capi.PLANE_VMAP), plane(1, capi.PLANE_NMAP), plane(0, capi.PLANE_VMAP),
                                 plane(0, capi.PLANE_NMAP), width, height, capi.ptr(pose), ctypes.byref(K),
                                 capi.ptr(scratch), capi.ptr(out), capi.stream_ptr()))
    out = out.cpu().numpy()
    assert sums[28] == out[28] > 0
    assert np.isclose(sums[27], out[27], rtol=1e-4)


@pytest.mark.parametrize("precision", [FP32, MIXED])
def test_batch_tracking_workgroups(precision):
    """A system's poses do not depend on the workgroups (1, 65, 300 or 512 partial rows) beyond the FP64 order of
    its sums."""
    from libfusion_amd.synth import Scene
    sc = Scene(1, 7)
    w, h = 640, 480
    K = capi.intrinsics(w, h, sc.fx, sc.fy, sc.cx, sc.cy)
    frames = [tuple(dev(a.view(np.int16) if a.dtype == np.uint16 else a) for a in sc.frame(i)) for i in range(3)]
    p = capi.map_params(1 << 18, 1 << 15, 0.01, 0.03, precision=precision)
    torch.cuda.synchronize()
    poses = []
    for wgs in (0, 1, 65, 300, 512):
        b = capi.Batch([capi.system_config(K, p, 3, (4, 3, 3), sc.depth_scale)])
        b.set_option(capi.BATCH_OPT_TRACK_WORKGROUPS, wgs)
        for d, c in frames:
            b.process([d], [c])
        b.synchronize()
        poses.append(b.pose(0))
        assert b.tracking(0)[0]
        b.close()
    # sums in another order differ by 1e-13 of their terms; a pose that enters the next step rounded to float32
    # another way moves it by up to 1e-7 of its 1.5 m
    for q in poses[1:]:
        assert np.allclose(q, poses[0], rtol=0, atol=3e-7)


# one workgroup, a partly filled one, 67 and 258 workgroups (past 64 and 256 rows), the capped grid on a ragged image
@pytest.mark.parametrize("width,height", [(16, 16), (19, 27), (184, 184), (363, 363), (641, 479)])
def test_reductions_in_one_launch(width, height):
    """The stand-alone reductions on scratch that holds anything, called again and again and replayed from a graph."""
    from oracle import oracle as O
    f = 525.0 * width / 640
    K = capi.intrinsics(width, height, f, f, (width - 1) / 2, (height - 1) / 2)
    oK = O.make_intr(K.width, K.height, K.fx, K.fy, K.cx, K.cy)
    maps = []
    for v, c in frame_pair(K, width, height):
        v = v.cpu().numpy()
        I = O.grey(c.cpu().numpy())
        maps.append((v, O.nmap(v), I) + tuple(O.derivative(I)))
    (lv, ln, lI, _, _), (cv, cn, cI, cdx, cdy) = maps
    t = [dev(a) for a in (cv, cn, lv, ln, cI, lI, cdx, cdy)]
    P, lib = capi.ptr, capi.load()
    n = lib.lf_reduce_scratch_floats()
    scratch = torch.randint(-2 ** 31, 2 ** 31 - 1, (n,), dtype=torch.int32, device="cuda").view(torch.float32)
    pose, icp, rgb = torch.empty(12, device="cuda"), torch.empty(29, device="cuda"), torch.empty(29, device="cuda")

    def call():
        st = capi.stream_ptr()
        capi.check(lib.lf_icp_reduce(P(t[0]), P(t[1]), P(t[2]), P(t[3]), width, height, P(pose), ctypes.byref(K),
                                     P(scratch), P(icp), st))
        capi.check(lib.lf_rgb_step(P(t[4]), P(t[5]), P(t[2]), P(t[6]), P(t[7]), width, height, 5.0, P(pose),
                                   ctypes.byref(K), P(scratch), P(rgb), st))

    def check(p12):
        # gates decided as by the float oracle; float32 sums of at most 2^19 terms against its FP64 ones
        for got, o in ((icp, lambda dt: O.icp_reduce(cv, cn, lv, ln, p12, oK, dt)),
                       (rgb, lambda dt: O.rgb_step(cI, lI, lv, cdx, cdy, np.float32(5.0), p12, oK, dt))):
            g, o32, o64 = got.cpu().numpy().astype(np.float64), o(np.float32).astype(np.float64), o(np.float64)
            assert g[28] == o32[28]
            assert np.allclose(g, o32, rtol=1e-4, atol=1e-5 * np.abs(o32).max())
            if o32[28] > 1000 and o32[28] == o64[28]:
                assert np.allclose(g, o64, rtol=1e-3, atol=1e-4 * np.abs(o64).max())

    poses = [np.eye(4)[:3].astype(np.float32).ravel() for _ in range(3)]
    for k, p in enumerate(poses):
        p[3] = 0.004 * k
    side = torch.cuda.Stream()
    for p in poses:
        pose.copy_(dev(p))
        call()
        check(p)
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        call()
    for p in poses:
        pose.copy_(dev(p))
        icp.fill_(-1)
        rgb.fill_(-1)
        g.replay()
        check(p)
        call()
        check(p)


# random depths under a band of 8 and of 50 voxels: a 16x16 tile requests a few hundred blocks, and more than its
# LDS set of 1024 holds; an image smaller than a tile and one with partial tiles
@pytest.mark.parametrize("precision", [FP32, MIXED])
@pytest.mark.parametrize("width,height,band", [(15, 9, 8), (72, 41, 8), (72, 41, 50)])
def test_allocation_of_scattered_requests(precision, width, height, band):
    """Allocated and visible blocks are the oracle's, and a de-integration lists the blocks the update did."""
    from oracle import oracle as O
    rng = np.random.default_rng(5)
    f = 525.0 * width / 640
    K = capi.intrinsics(width, height, f, f, (width - 1) / 2, (height - 1) / 2)
    depth = rng.uniform(0.4, 4.8, (height, width)).astype(np.float32)
    depth[rng.random(depth.shape) < 0.05] = 0.0
    nmap = np.zeros((height, width, 4), np.float32)
    nmap[..., 2] = 1.0
    rgb = rng.integers(0, 256, (height, width, 3)).astype(np.uint8)
    T = np.eye(4)
    T[:3, 3] = (0.3, -0.2, 0.1)
    p = capi.map_params(1 << 16, 1 << 16, 0.004, 0.004 * band, precision=precision)
    m = capi.Map(p, max(width, 8), max(height, 8))
    pose = dev(capi.pose24(T))
    m.update_weighted(dev(depth), dev(nmap), dev(rgb), pose, K)
    om = O.Map(O.Params(p.num_buckets, p.num_entries, p.num_blocks, p.max_triangles, p.zmin_raycast, p.zmax_raycast,
                        p.zmin_update, p.zmax_update, p.voxel_size, p.truncation), np.float32)
    om.update_weighted(depth, nmap, rgb, T, O.make_intr(K.width, K.height, K.fx, K.fy, K.cx, K.cy))
    key = lambda b: set(map(tuple, b.tolist()))  # noqa: E731
    got, want = key(m.blocks()), key(om.blocks())
    if precision == FP32:
        assert got == want
    else:  # a product with the reciprocal voxel size moves band ends that lie on a block face
        assert len(got ^ want) <= max(2, len(want) // 200)
    seen = key(m.visible_blocks())
    assert seen == got  # every requested block is listed
    n = int(m.counters()[capi.CNT_ALLOCATED])
    m.deintegrate_weighted(dev(depth), dev(nmap), dev(rgb), pose, K)
    assert key(m.visible_blocks()) == seen and int(m.counters()[capi.CNT_ALLOCATED]) == n
    assert not m.t["slot_flag"].any()


# images of 1 to 2 pixels, of odd sizes, and of more blocks than the launch's workgroups
@pytest.mark.parametrize("width,height,dist", [(1, 1, 1.0), (2, 1, 1.0), (33, 7, 0.7), (161, 121, 1.5)])
def test_separate_planes_fuse_and_take_out(width, height, dist):
    """A frame fused and taken out from depth, normal and colour planes, against the updates restated in numpy.

    The projections are the same float32 operations, so both pick the same pixels; a weight differs by sin's last
    bits (1e-6 of it), a code or a colour by one where that moves a quotient past a whole number."""
    rng = np.random.default_rng(11)
    f32 = np.float32
    f = 525.0 * max(width, 16) / 640
    K = capi.intrinsics(width, height, f, f, (width - 1) / 2, (height - 1) / 2)
    T = np.eye(4)
    T[:3, 3] = (0.013, -0.007, 0.011)
    a = 0.05
    T[:3, :3] = [[np.cos(a), 0, np.sin(a)], [0, 1, 0], [-np.sin(a), 0, np.cos(a)]]
    p24 = capi.pose24(T)
    vs, trunc = f32(0.01), f32(0.03)
    p = capi.map_params(1 << 14, 1 << 14, float(vs), float(trunc))
    m = capi.Map(p, max(width, 8), max(height, 8))

    def frame(lo, hi):
        depth = (dist + rng.uniform(-0.02, 0.02, (height, width))).astype(f32)
        nmap = rng.uniform(lo, hi, (height, width, 4)).astype(f32)
        if width * height > 4:
            depth[rng.random(depth.shape) < 0.05] = np.nan
            nmap[rng.random(depth.shape) < 0.05, 0] = np.nan
        return depth, nmap, rng.integers(0, 256, (height, width, 3)).astype(np.uint8)

    def observe(blocks, fr):
        depth, nmap, rgb = fr
        q = np.arange(512)
        w = [(blocks[:, k, None] * 8 + (q >> (3 * k) & 7)).astype(f32) * vs for k in range(3)]
        M = p24[12:].reshape(3, 4)
        c = [M[k, 0] * w[0] + M[k, 1] * w[1] + M[k, 2] * w[2] + M[k, 3] for k in range(3)]
        with np.errstate(all="ignore"):
            tu = f32(K.fx) * c[0] / c[2] + f32(K.cx) + f32(0.5)
            tv = f32(K.fy) * c[1] / c[2] + f32(K.cy) + f32(0.5)
        ok = (tu >= 0) & (tu < width) & (tv >= 0) & (tv < height)
        u, v = np.where(ok, tu, 0).astype(int), np.where(ok, tv, 0).astype(int)
        d, n = depth[v, u], nmap[v, u]
        s = d - c[2]
        with np.errstate(invalid="ignore"):
            ok &= (d <= f32(p.zmax_update)) & (d >= f32(p.zmin_update)) & ~np.isnan(n[..., 0]) & ~(s < -trunc)
        s = np.minimum(f32(1), s * f32(f32(1) / trunc))
        return ok, s, np.abs(np.sin(n[..., 2])) / (d * d), rgb[v, u].transpose(0, 2, 1).astype(f32)

    def step(fr, take_out):
        planes = [dev(x) for x in fr]
        before = {tuple(b): i for i, b in enumerate(m.blocks().tolist())}
        _, s0, w0, c0 = m.voxels()
        (m.deintegrate_weighted if take_out else m.update_weighted)(*planes, dev(p24), K)
        torch.cuda.synchronize()
        blocks, s1, w1, c1 = m.voxels()
        n = len(blocks)
        assert n > 0 and [before.get(tuple(b), i) for i, b in enumerate(blocks.tolist())] == list(range(n))
        grow = lambda x: np.concatenate([x, np.zeros((n - len(x),) + x.shape[1:], x.dtype)])  # noqa: E731
        codes, w0, c0 = grow(s0), grow(w0), grow(c0).astype(f32)
        seen = {tuple(b) for b in m.visible_blocks().tolist()}
        ok, s, w, col = observe(blocks, fr)
        ok &= np.array([tuple(b) in seen for b in blocks.tolist()])[:, None]
        s0 = codes.astype(f32) / f32(32767)
        with np.errstate(all="ignore"):
            if take_out:
                ok &= w0 != 0
                wn = w0 - w
                sn = np.clip((s0 * w0 - s * w) / wn, -1, 1)
                cn = np.clip((c0 * w0[:, None] - col * w[:, None]) / wn[:, None], 0, 255)
                gone = ok & (wn <= 0)
                sn, wn, cn = (np.where(g, 0, x) for g, x in ((gone, sn), (gone, wn), (gone[:, None], cn)))
            else:
                wn = w0 + w
                sn = np.where(w0 == 0, s, (s0 * w0 + s * w) / wn)
                cn = np.where(w0[:, None] == 0, col, (c0 * w0[:, None] + col * w[:, None]) / wn[:, None])
        assert ok.any()
        sn, cn = np.trunc(np.where(ok, sn, s0) * f32(32767)), np.trunc(np.where(ok[:, None], cn, c0))
        wn = np.where(ok, wn, w0)
        assert np.all(np.abs(w1 - wn) <= 4e-6 * np.maximum(w0, wn))
        sure = np.abs(wn) > 1e-3 * w0  # the rest of a weight that all but cancels is rounding
        ratio = np.maximum(1, w0 / np.maximum(wn, 1e-30))
        assert np.all((np.abs(s1 - sn) <= 1 + 0.1 * ratio)[sure & (wn > 0)])
        assert np.all((np.abs(c1 - cn) <= (1 + 1e-3 * ratio)[:, None]).transpose(0, 2, 1)[sure & (wn > 0)])
        assert np.array_equal(s1[~ok], codes[~ok]) and np.array_equal(w1[~ok], w0[~ok])

    first, second, third = frame(0.1, 0.3), frame(0.4, 1.0), frame(0.4, 1.0)
    step(first, False)
    step(second, False)
    step(second, True)
    step(third, True)  # heavier than what is left: the voxels return to unseen
    assert (m.voxels()[2] == 0).any()


# one level of odd size and of one pixel; levels of one pixel; partial tiles on every level; more levels than the
# first passes hold
@pytest.mark.parametrize("width,height,levels", [(1, 1, 1), (37, 5, 1), (2, 2, 2), (46, 18, 2), (4, 4, 3),
                                                 (72, 40, 3), (72, 40, 4), (160, 96, 6)])
def test_image_passes(width, height, levels):
    """upload and resize_device_map store what the operations one at a time give, bit for bit, from a colour image
    at an odd address too."""
    rng = np.random.default_rng(3)
    lib, st, P = capi.load(), capi.stream_ptr(), capi.ptr
    f = 525.0 * width / 640
    K = capi.intrinsics(width, height, f, f, (width - 1) / 2, (height - 1) / 2)
    img = capi.Image(K, levels)
    d16 = rng.integers(0, 6000, (height, width)).astype(np.uint16)
    scale = float(np.float32(1e-3))
    colours = dev(rng.integers(0, 256, 3 * width * height + 1).astype(np.uint8))
    d16_t, rgb_t = dev(d16), colours[1:]
    img.upload(d16_t, rgb_t, scale)
    like = lambda l, *c: torch.empty((img.K[l].height, img.K[l].width) + c, device="cuda")  # noqa: E731

    def same(l, plane, ref):
        assert np.array_equal(img.plane(l, plane).cpu().numpy(), ref.cpu().numpy(), equal_nan=True), (l, plane)

    def normals(vm, l):
        n = like(l, 4)
        capi.check(lib.lf_compute_nmap(P(vm), P(n), img.K[l].width, img.K[l].height, st))
        return n

    raw, depth, grey = like(0), [like(l) for l in range(levels)], [like(l) for l in range(levels)]
    capi.check(lib.lf_depth_to_float(P(d16_t), P(raw), width, height, scale, st))
    capi.check(lib.lf_bilateral_filter(P(raw), P(depth[0]), width, height, st))
    capi.check(lib.lf_rgb_to_intensity(P(rgb_t), P(grey[0]), width, height, st))
    same(0, capi.PLANE_RAW_DEPTH, raw)
    same(0, capi.PLANE_RGB, rgb_t.view(height, width, 3))
    for l in range(levels):
        w, h = img.K[l].width, img.K[l].height
        if l:
            capi.check(lib.lf_pyr_down_depth(P(depth[l - 1]), P(depth[l]), 2 * w, 2 * h, st))
            capi.check(lib.lf_pyr_down_image(P(grey[l - 1]), P(grey[l]), 2 * w, 2 * h, st))
        dx, dy, vm = like(l), like(l), like(l, 4)
        capi.check(lib.lf_compute_derivative(P(grey[l]), P(dx), P(dy), w, h, st))
        capi.check(lib.lf_back_project_depth(P(depth[l]), P(vm), w, h, ctypes.byref(img.K[l]), st))
        for plane, ref in ((capi.PLANE_DEPTH, depth[l]), (capi.PLANE_INTENSITY, grey[l]), (capi.PLANE_DX, dx),
                           (capi.PLANE_DY, dy), (capi.PLANE_VMAP, vm), (capi.PLANE_NMAP, normals(vm, l))):
            same(l, plane, ref)
    v = dev(rng.uniform(-1, 4, (height, width, 4)).astype(np.float32))
    torch.cuda.synchronize()
    capi.copy_device_to(img.plane_ptr(0, capi.PLANE_VMAP), v)
    img.resize_device_map()
    for l in range(levels):
        if l:
            half = like(l, 4)
            capi.check(lib.lf_pyr_down_vmap(P(v), P(half), img.K[l - 1].width, img.K[l - 1].height, st))
            v = half
        same(l, capi.PLANE_VMAP, v)
        same(l, capi.PLANE_NMAP, normals(v, l))
    img.close()


# the block directory ends 5.12 m from the origin on each axis: views inside it, across its faces, its corner, outside;
# a step of 1.5 and of 25 voxels
@pytest.mark.parametrize("band", [3, 50])
@pytest.mark.parametrize("at", [(0.0, 0.0, 0.0), (5.0, 0.2, -0.5), (-5.1, 0.0, 1.0), (0.1, 5.08, 0.0), (0.0, 0.0, 4.2),
                                (-4.95, -5.05, 4.3), (7.0, -6.5, 6.0)])
def test_raycast_around_the_directory(at, band):
    """Vertices and colours of a rough surface with holes, bit for bit the oracle's on the same volume."""
    from oracle import oracle as O
    rng = np.random.default_rng(17)
    width, height = 72, 41
    f = 525.0 * width / 640
    K = capi.intrinsics(width, height, f, f, (width - 1) / 2, (height - 1) / 2)
    u, v = np.meshgrid(np.linspace(0, 7, width), np.linspace(0, 4, height))
    depth = (0.9 + 0.2 * np.sin(u) * np.cos(v) + 0.01 * rng.random((height, width))).astype(np.float32)
    depth[rng.random(depth.shape) < 0.1] = 0.0
    depth[10:20, 30:40] += 0.5
    nmap = np.zeros((height, width, 4), np.float32)
    nmap[..., 2] = 1.0
    rgb = rng.integers(0, 256, (height, width, 3)).astype(np.uint8)
    a, b = 0.3, -0.2
    T = np.eye(4)
    T[:3, :3] = (np.array([[np.cos(a), 0, np.sin(a)], [0, 1, 0], [-np.sin(a), 0, np.cos(a)]])
                 @ np.array([[1, 0, 0], [0, np.cos(b), -np.sin(b)], [0, np.sin(b), np.cos(b)]]))
    T[:3, 3] = at
    p = capi.map_params(1 << 16, 1 << 15, 0.005, 0.005 * band)
    m = capi.Map(p, width, height)
    pose = dev(capi.pose24(T))
    m.update_weighted(dev(depth), dev(nmap), dev(rgb), pose, K)
    vm = torch.full((height, width, 4), float("nan"), device="cuda")
    col = torch.zeros((height, width, 3), dtype=torch.uint8, device="cuda")
    m.raycast(vm, pose, K, check_colour=True, rgb_out=col)
    torch.cuda.synchronize()
    om = O.Map(O.Params(p.num_buckets, p.num_entries, p.num_blocks, p.max_triangles, p.zmin_raycast, p.zmax_raycast,
                        p.zmin_update, p.zmax_update, p.voxel_size, p.truncation), np.float32)
    oK = O.make_intr(K.width, K.height, K.fx, K.fy, K.cx, K.cy)
    om.update_weighted(depth, nmap, rgb, T, oK)
    om.set_blocks(*m.voxels())
    ovm, ocol = om.raycast(T, oK, width, height, check_colour=True, want_rgb=True)
    hit = ~np.isnan(ovm[..., 0])
    assert hit.mean() > 0.4
    assert np.array_equal(vm.cpu().numpy()[hit], ovm[hit]) and np.isnan(vm.cpu().numpy()[~hit]).all()
    assert np.array_equal(col.cpu().numpy(), ocol)


# an image inside one tile, partial tiles, and blocks that span more tiles than the depth test looks at
@pytest.mark.parametrize("width,height,voxel", [(7, 5, 0.01), (61, 43, 0.01), (64, 48, 0.01), (160, 120, 0.02)])
def test_refusion_with_occlusions(width, height, voxel):
    """Keyframes of patches at depths that hide each other, none and out of range among them: re-fusion leaves the
    voxels seen, and their weights, that one keyframe after the other does (the same float weight arithmetic)."""
    rng = np.random.default_rng(23)
    f = 525.0 * max(width, 32) / 640
    K = capi.intrinsics(width, height, f, f, (width - 1) / 2, (height - 1) / 2)
    p = capi.map_params(1 << 17, 1 << 16, voxel, 3 * voxel)
    n = 6
    imgs, old, new = [], [], []

    def pose():
        T = np.eye(4)
        a = rng.uniform(-0.3, 0.3)
        T[:3, :3] = [[np.cos(a), 0, np.sin(a)], [0, 1, 0], [-np.sin(a), 0, np.cos(a)]]
        T[:3, 3] = rng.uniform(-0.2, 0.2, 3)
        return T

    for _ in range(n):
        patches = rng.choice([0, 500, 800, 1200, 1900, 2600, 9000], (height // 6 + 1, width // 9 + 1))
        d16 = np.kron(patches, np.ones((6, 9), int))[:height, :width] + rng.integers(0, 4, (height, width))
        img = capi.Image(K, 1)
        img.upload(dev(d16.astype(np.uint16)), dev(rng.integers(0, 256, (height, width, 3)).astype(np.uint8)), 1e-3)
        T = pose()
        imgs.append(img)
        old.append(dev(capi.pose24(T)))
        T[:3, 3] += rng.uniform(-0.02, 0.02, 3)
        new.append(dev(capi.pose24(T)))
    base, seq, one = (capi.Map(p, max(width, 8), max(height, 8)) for _ in range(3))
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
    bo, _, wo, _ = one.voxels()
    bs, _, ws, _ = seq.voxels()
    at = {tuple(b): i for i, b in enumerate(bo.tolist())}
    assert set(map(tuple, bs.tolist())) == set(at) and (ws > 0).sum() > 50
    assert np.array_equal(wo[[at[tuple(b)] for b in bs.tolist()]], ws)
    for img in imgs:
        img.close()


@pytest.mark.parametrize("width,height,levels", [(1, 1, 1), (37, 5, 1), (2, 2, 2), (46, 18, 2), (4, 4, 3),
                                                 (72, 40, 3), (160, 96, 6)])
@pytest.mark.parametrize("offset", [0, 1])
def test_tracker_planes(width, height, levels, offset):
    """set_*_image, set_*_intensity and set_*_vmap store what the operations one at a time give, bit for bit, from
    planes at unaligned addresses too (offset floats, or bytes, into their buffer)."""
    rng = np.random.default_rng(7)
    lib, st, P = capi.load(), capi.stream_ptr(), capi.ptr
    f = 525.0 * width / 640
    tr = capi.Tracker(capi.intrinsics(width, height, f, f, (width - 1) / 2, (height - 1) / 2), levels)
    n = width * height
    rgb = dev(rng.integers(0, 256, 3 * n + offset).astype(np.uint8))[offset:]
    grey = dev(rng.uniform(0, 255, n + offset).astype(np.float32))[offset:]
    vmap = dev(rng.uniform(-1, 4, 4 * n + offset).astype(np.float32))[offset:]

    def same(source, l, which, ref):
        out = ctypes.c_void_p()
        capi.check(lib.lf_tracker_plane(tr.h, source, l, which, ctypes.byref(out)))
        t = torch.empty_like(ref)
        capi.copy_device(t, out.value, t.numel() * t.element_size())
        assert np.array_equal(t.cpu().numpy(), ref.cpu().numpy(), equal_nan=True), (source, l, which)

    tr.set("set_source_image", rgb)
    tr.set("set_reference_intensity", grey)
    tr.set("set_reference_vmap", vmap)
    first = torch.empty(height, width, device="cuda")
    capi.check(lib.lf_rgb_to_intensity(P(rgb), P(first), width, height, st))
    for source, plane in ((1, first), (0, grey.view(height, width).clone())):
        for l in range(levels):
            w, h = tr.K[l].width, tr.K[l].height
            if l:
                half = torch.empty(h, w, device="cuda")
                capi.check(lib.lf_pyr_down_image(P(plane), P(half), 2 * w, 2 * h, st))
                plane = half
            dx, dy = torch.empty_like(plane), torch.empty_like(plane)
            capi.check(lib.lf_compute_derivative(P(plane), P(dx), P(dy), w, h, st))
            for which, ref in ((capi.PLANE_INTENSITY, plane), (capi.PLANE_DX, dx), (capi.PLANE_DY, dy)):
                if source or which == capi.PLANE_INTENSITY:
                    same(source, l, which, ref)
    v = vmap.view(height, width, 4).clone()
    for l in range(levels):
        w, h = tr.K[l].width, tr.K[l].height
        if l:
            half = torch.empty(h, w, 4, device="cuda")
            capi.check(lib.lf_pyr_down_vmap(P(v), P(half), 2 * w, 2 * h, st))
            v = half
        nm = torch.empty_like(v)
        capi.check(lib.lf_compute_nmap(P(v), P(nm), w, h, st))
        same(0, l, capi.PLANE_VMAP, v)
        same(0, l, capi.PLANE_NMAP, nm)
    tr.close()


# none, far below the first normal code's 2^-6, on both sides of it, ordinary, large
@pytest.mark.parametrize("weight", [0.0, 3e-4, 0.0155, 0.0157, 0.5, 6.0])
def test_mixed_weights_and_colours(weight):
    """A mixed map's words after two frames of one depth, weight and colour each: the weight codes are
    lf_weight_code_dither of the summed weights with the voxel's random bits (but for the sum's last bit: one code at a
    few voxels), the colours the truncated means (one level either side, by the mean's rounding)."""
    rng = np.random.default_rng(2)
    width, height, d = 40, 30, np.float32(0.4)
    K = capi.intrinsics(width, height, 40.0, 40.0, (width - 1) / 2, (height - 1) / 2)
    p = capi.map_params(1 << 12, 1 << 12, 0.01, 0.03, precision=MIXED)
    m = capi.Map(p, width, height)
    pose = dev(capi.pose24(np.eye(4)))
    lib = capi.load()
    value = lambda c: c / 1024 if c < 16 else (1 + (c & 15) / 16) * 2.0 ** ((c >> 4) - 7)  # noqa: E731
    values = np.array([value(c) for c in range(256)], np.float32)

    def words():
        n = int(m.counters()[capi.CNT_ALLOCATED])
        w = m.t["weight"][: 512 * n].view(n, 512).cpu().numpy().view(np.uint32)
        return m.blocks().astype(np.int64), w & 0xFF, np.stack([w >> (8 + 8 * k) & 0xFF for k in range(3)], -1)

    def fuse(wt, rgb):
        nmap = np.zeros((height, width, 4), np.float32)
        nmap[..., 2] = np.arcsin(np.float64(wt) * np.float64(d) ** 2)
        m.update_weighted(dev(np.full((height, width), d)), dev(nmap),
                          dev(np.full((height, width, 3), rgb, np.uint8)), pose, K)
        torch.cuda.synchronize()

    def random_bits(blocks, i, l):
        x, y, z = (blocks[i, k] * c & 0xFFFFFFFF for k, c in enumerate((0x9E3779B1, 0x85EBCA77, 0xC2B2AE3D)))
        r = x ^ y ^ z ^ ((l + (int(m.counters()[8]) << 9)) * 0x27D4EB2F & 0xFFFFFFFF)
        r ^= r >> 16
        r = r * 0x7FEB352D & 0xFFFFFFFF
        r ^= r >> 15
        r = r * 0x846CA68B & 0xFFFFFFFF
        return r ^ r >> 16

    def check(at, codes, sums):
        blocks, i, l = at
        want = np.array([lib.lf_weight_code_dither(float(s), int(r))
                         for s, r in zip(sums, random_bits(blocks, i, l))])
        off = np.abs(codes[i, l].astype(int) - np.maximum(want, 1))
        assert off.max() <= 1 and (off > 0).mean() < 0.01, (off.max(), (off > 0).mean())

    first, second, wt2 = rng.integers(0, 256, 3), rng.integers(0, 256, 3), np.float32(0.3)
    fuse(weight, first)
    blocks, c1, col1 = words()
    if weight == 0.0:
        assert not c1.any()
        fuse(wt2, second)
        blocks, c1, col1 = words()
        first, weight = second, wt2
    i, l = np.nonzero(c1)
    assert len(i) > 5000 and (col1[i, l] == first).all()
    check((blocks, i, l), c1, np.full(len(i), np.float32(weight)))
    fuse(wt2, second)
    again, c2, col2 = words()
    assert np.array_equal(again[: len(blocks)], blocks)
    w1 = values[c1[i, l]]
    check((again, i, l), c2, np.minimum(w1 + wt2, np.float32(255)))
    mean = (w1[:, None].astype(np.float64) * first + np.float64(wt2) * second) / (w1[:, None].astype(np.float64) + wt2)
    assert np.all(np.abs(col2[i, l] - np.floor(mean)) <= 1)


def test_state_reads_from_several_threads():
    """A System's pose and tracking result, read by threads at once beside the frames enqueued, are the serial reads'."""
    from concurrent.futures import ThreadPoolExecutor
    rng = np.random.default_rng(1)
    K = capi.intrinsics(64, 48, 52.5, 52.5, 31.5, 23.5)
    s = capi.System(K, capi.map_params(1 << 12, 1 << 12, 0.02, 0.06), 2, (3, 2), 1e-3)
    u, v = np.meshgrid(np.linspace(0, 6, 64), np.linspace(0, 4, 48))
    for f in range(3):
        d16 = (1000 + 150 * np.sin(u + 0.01 * f) * np.cos(v)).astype(np.uint16)
        s.process(dev(d16), dev(rng.integers(0, 256, (48, 64, 3)).astype(np.uint8)))
        with ThreadPoolExecutor(4) as pool:
            poses = list(pool.map(lambda _: s.pose(), range(8)))
            results = list(pool.map(lambda _: s.tracking(), range(8)))
        assert all(np.array_equal(p, s.pose()) for p in poses)
        assert all(np.array_equal(r, s.tracking(), equal_nan=True) for r in results)  # a lost frame has no error


# one workgroup, one per XCD and one more, the last grid whose workgroups are resident at once and the first that isn't
@pytest.mark.parametrize("width,height", [(16, 8), (128, 16), (144, 16), (1024, 512), (1040, 512)])
def test_raycast_grids(width, height):
    """Every pixel of a raycast is the oracle's, bit for bit, whichever XCD takes its tile."""
    from oracle import oracle as O
    f = 0.8 * width
    K = capi.intrinsics(width, height, f, f, (width - 1) / 2, (height - 1) / 2)
    u, v = np.meshgrid(np.linspace(0, 9, width), np.linspace(0, 5, height))
    depth = (0.8 + 0.1 * np.sin(u) * np.cos(v)).astype(np.float32)
    nmap = np.zeros((height, width, 4), np.float32)
    nmap[..., 2] = 1.0
    rgb = np.full((height, width, 3), 77, np.uint8)
    T = np.eye(4)
    p = capi.map_params(1 << 16, 1 << 15, 0.01, 0.03)
    m = capi.Map(p, width, height)
    pose = dev(capi.pose24(T))
    m.update_weighted(dev(depth), dev(nmap), dev(rgb), pose, K)
    vm = torch.full((height, width, 4), -1.0, device="cuda")
    m.raycast(vm, pose, K)
    torch.cuda.synchronize()
    om = O.Map(O.Params(p.num_buckets, p.num_entries, p.num_blocks, p.max_triangles, p.zmin_raycast, p.zmax_raycast,
                        p.zmin_update, p.zmax_update, p.voxel_size, p.truncation), np.float32)
    oK = O.make_intr(K.width, K.height, K.fx, K.fy, K.cx, K.cy)
    om.update_weighted(depth, nmap, rgb, T, oK)
    om.set_blocks(*m.voxels())
    ovm = om.raycast(T, oK, width, height)
    assert (~np.isnan(ovm[..., 0])).mean() > 0.5
    assert np.array_equal(vm.cpu().numpy(), ovm, equal_nan=True)


# one tile; a workgroup's box one narrower, as wide and one wider than the 32 lanes of its rows; the grid that just fits
# LDS; one that doesn't
@pytest.mark.parametrize("width,height", [(8, 8), (248, 120), (256, 256), (264, 272), (1280, 960), (1600, 1040)])
def test_zrange_tiles(width, height):
    """Each tile's depth range is the oracle's, bit for bit, however many workgroups and passes share it."""
    from oracle import oracle as O
    f = 0.8 * width
    K = capi.intrinsics(width, height, f, f, (width - 1) / 2, (height - 1) / 2)
    u, v = np.meshgrid(np.linspace(0, 9, width), np.linspace(0, 5, height))
    depth = (0.8 + 0.1 * np.sin(u) * np.cos(v)).astype(np.float32)
    nmap = np.zeros((height, width, 4), np.float32)
    nmap[..., 2] = 1.0
    rgb = np.full((height, width, 3), 77, np.uint8)
    T = np.eye(4)
    p = capi.map_params(1 << 16, 1 << 15, 0.005, 0.015)
    m = capi.Map(p, width, height)
    pose = dev(capi.pose24(T))
    m.update_weighted(dev(depth), dev(nmap), dev(rgb), pose, K)
    m.raycast(torch.empty((height, width, 4), device="cuda"), pose, K)
    torch.cuda.synchronize()
    om = O.Map(O.Params(p.num_buckets, p.num_entries, p.num_blocks, p.max_triangles, p.zmin_raycast, p.zmax_raycast,
                        p.zmin_update, p.zmax_update, p.voxel_size, p.truncation), np.float32)
    oK = O.make_intr(K.width, K.height, K.fx, K.fy, K.cx, K.cy)
    om.update_weighted(depth, nmap, rgb, T, oK)
    near, far = om.zrange(T, oK, width, height)
    tiles = (width // 8) * (height // 8)
    got = m.t["zrange"].cpu().numpy()
    assert (near < 100).mean() > 0.9
    assert np.array_equal(got[:tiles], near.ravel()) and np.array_equal(got[tiles : 2 * tiles], far.ravel())


@pytest.mark.parametrize("precision", [FP32, MIXED])
@pytest.mark.parametrize("n", [1, 2])
def test_batch_raycast_grids(n, precision):
    """Maps dealt to the XCDs by bands where few (1500 workgroups) and a few tiles at a time where many (2700): the
    poses tracked against their raycasts are those of each map alone."""
    from libfusion_amd.synth import Scene
    cfgs, frames = [], []
    for div in [1] * n + [2]:
        sc = Scene(1, 7)
        K = capi.intrinsics(sc.width // div, sc.height // div, sc.fx / div, sc.fy / div, (sc.cx + 0.5) / div - 0.5,
                            (sc.cy + 0.5) / div - 0.5)
        p = capi.map_params(1 << 18, 1 << 15, 0.01, 0.03, precision=precision)
        cfgs.append(capi.system_config(K, p, 2, (4, 3), sc.depth_scale))
        shots = [sc.render(sc.pose(i), K.width, K.height, K.fx, K.fy, K.cx, K.cy, noise=True, frame_id=i)
                 for i in range(3)]
        frames.append([(dev(d.view(np.int16)), dev(c)) for d, c in shots])
    torch.cuda.synchronize()

    def run(which):
        b = capi.Batch([cfgs[i] for i in which])
        for t in range(3):
            b.process([frames[i][t][0] for i in which], [frames[i][t][1] for i in which])
        b.synchronize()
        assert all(b.tracking(k)[0] for k in range(len(which)))
        poses = [b.pose(k) for k in range(len(which))]
        b.close()
        return poses

    together = run(range(n + 1))
    for i in (0, n):
        # the tracking sums of 1 / n of the workgroups in another order: see test_batch_tracking_workgroups
        assert np.allclose(together[i], run([i])[0], rtol=0, atol=3e-7), i
