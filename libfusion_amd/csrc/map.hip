// Voxel-hash block allocation, visible-block selection and TSDF integration.
//
// Reference: src/voxel_hashing/depth_fusion.cu (create_blocks_kernel :121-228,
// check_visibility_flag_kernel :49-83, copy_visible_block_kernel :85-93,
// update_map_kernel / update_map_with_colour_kernel / update_map_weighted_kernel
// :230-428, host update / update_weighted :430-575) and the hash-map primitives
// of src/data_struct/map_struct.cu (computeHash :143-148, createBlock :280-325,
// findEntry :365-381).
//
// MI355X design (not a translation of the reference's scheme):
//  * The table is open addressing with linear probing from computeHash's home
//    bucket over num_entries slots.  A slot holds a 63-bit packed block
//    coordinate claimed with one 64-bit CAS — no bucket locks, so no request is
//    ever dropped (the reference drops an allocation when a bucket lock is
//    contended, map_struct.cu:303-324).
//  * Pool blocks are handed out by an atomic counter and their coordinates are
//    recorded in allocation order (block_pos), so visibility runs over the
//    allocated blocks, O(allocated), instead of scanning every table entry.
//  * A 16x16-pixel workgroup first deduplicates its requests in an LDS hash set
//    (ds_cmpst_b64): neighbouring pixels request the same few blocks, so only
//    unique keys reach HBM.
//  * The visible list is appended with one atomic per workgroup (ballots, the
//    wavefronts' counts prefixed in LDS).
//  * Integration walks the visible list with a fixed grid (grid-stride), one
//    256-thread workgroup per 8^3 block: each lane owns two voxels of the
//    block's contiguous 512-voxel run, so every voxel plane is read and written
//    with fully coalesced 128-byte wavefront accesses.
#include "lf_common.h"
#include "lf_internal.h"

using namespace lf;

namespace {

struct MapDev {
    unsigned long long *keys;
    int *slot_block;
    unsigned char *slot_flag;
    int *block_pos;
    short *sdf;
    float *weight;
    unsigned char *rgb;
    int *visible;
    int *visible_pos;  // {x, y, z, pool block} of visible[i]
    int *block_dir;    // LF_DIR_CELLS pool blocks, -1 = none
    unsigned int *counters;
    unsigned int *occupancy;
    int num_buckets, num_entries, num_blocks;
    float voxel_size, truncation, zmin_update, zmax_update;
    float inv_truncation;  // 1 / truncation, computed on the host (the same correctly rounded division)
};

// A map read from a descriptor table, its pointers asserted global.
LF_DEV MapDev global_dev(const MapDev &d) {
    MapDev m = d;
    m.keys = global_ptr(d.keys); m.slot_block = global_ptr(d.slot_block); m.slot_flag = global_ptr(d.slot_flag);
    m.block_pos = global_ptr(d.block_pos); m.sdf = global_ptr(d.sdf); m.weight = global_ptr(d.weight);
    m.rgb = global_ptr(d.rgb); m.visible = global_ptr(d.visible); m.visible_pos = global_ptr(d.visible_pos);
    m.block_dir = global_ptr(d.block_dir); m.counters = global_ptr(d.counters); m.occupancy = global_ptr(d.occupancy);
    return m;
}

MapDev make_dev(const lf_map_params *p, const lf_map_storage *s) {
    MapDev d;
    d.keys = s->keys; d.slot_block = s->slot_block; d.slot_flag = s->slot_flag; d.block_pos = s->block_pos;
    d.sdf = s->sdf; d.weight = s->weight; d.rgb = s->rgb; d.visible = s->visible; d.counters = s->counters;
    d.occupancy = s->occupancy;
    d.visible_pos = s->visible_pos;
    d.block_dir = s->block_dir;
    d.num_buckets = p->num_buckets; d.num_entries = p->num_entries; d.num_blocks = p->num_blocks;
    d.voxel_size = p->voxel_size; d.truncation = p->truncation;
    d.inv_truncation = 1.0f / p->truncation;
    d.zmin_update = p->zmin_update; d.zmax_update = p->zmax_update;
    return d;
}

// createBlock (map_struct.cu:280-325) as a lock-free insert.  Marks the slot as
// touched by this update (the reference's flag = 2, depth_fusion.cu:157).
// Returns the block's hash slot (-1: the table is full); *claimed: this call
// created the entry.
LF_DEV int insert_block(const MapDev &m, int bx, int by, int bz, bool *claimed_out = nullptr) {
    const unsigned long long key = pack_key(bx, by, bz);
    int slot = compute_hash(bx, by, bz, m.num_buckets);
    for (int i = 0; i < m.num_entries; ++i) {
        // A plain load may see a stale empty slot (another XCD's L2); the CAS is
        // authoritative.  A non-empty key never changes until the next reset.
        unsigned long long k = m.keys[slot];
        bool claimed = false;
        if (k == kEmptyKey) {
            k = atomicCAS(&m.keys[slot], kEmptyKey, key);
            claimed = (k == kEmptyKey);
        }
        if (claimed) {
            const unsigned int ob = occupancy_bit(bx, by, bz);
            atomicOr(&m.occupancy[ob >> 5], 1u << (ob & 31));
            unsigned int b = atomicAdd(&m.counters[LF_CNT_ALLOCATED], 1u);
            if (b < (unsigned int)m.num_blocks) {
                m.slot_block[slot] = (int)b;
                reinterpret_cast<int4 *>(m.block_pos)[b] = make_int4(bx, by, bz, slot);
                const int cell = dir_cell(bx, by, bz);
                if (cell >= 0) m.block_dir[cell] = (int)b;
            } else {
                atomicOr(&m.counters[LF_CNT_OVERFLOW], LF_OVF_POOL);
            }
            m.slot_flag[slot] = 1;
            if (claimed_out) *claimed_out = true;
            return slot;
        }
        if (k == key) {
            m.slot_flag[slot] = 1;
            return slot;
        }
        if (++slot == m.num_entries) slot = 0;
    }
    atomicOr(&m.counters[LF_CNT_OVERFLOW], LF_OVF_TABLE);
    return -1;
}

// One pixel of create_blocks_kernel (depth_fusion.cu:121-228): the 3-D
// Bresenham walk over the blocks between the near and far ends of the
// truncation band around the measured depth.  kFast (mixed precision): the
// voxel coordinates by a product with the reciprocal voxel size.
template <bool kFast, class F>
LF_DEV void band_blocks(int x, int y, float z, const float *Twc, const lf_intrinsics &K, const MapDev &m, F emit) {
    const float zmin = m.zmin_update, zmax = m.zmax_update;
    if (isnan(z) || z < zmin || z > zmax) return;
    const float half = m.truncation * 0.5f;
    const float zn = fmaxf(zmin, z - half);
    const float zf = fminf(zmax, z + half);
    if (zn >= zf) return;
    const float vs = m.voxel_size;
    const float ux = K.invfx * ((float)x - K.cx), uy = K.invfy * ((float)y - K.cy);
    f3 pn = xform(Twc, f3{ux * zn, uy * zn, zn});
    f3 pf = xform(Twc, f3{ux * zf, uy * zf, zf});
    i3 vn, vf;
    if (kFast) {
        const float iv = 1.0f / vs;
        vn = to_i3(mul(pn, iv));
        vf = to_i3(mul(pf, iv));
    } else {  // the divisions' floats (an infinite coordinate is refused either way)
        const Recip iv = recip(vs);
        vn = to_i3(f3{quotient(pn.x, iv), quotient(pn.y, iv), quotient(pn.z, iv)});
        vf = to_i3(f3{quotient(pf.x, iv), quotient(pf.y, iv), quotient(pf.z, iv)});
    }
    if (vn.x == kBad || vn.y == kBad || vn.z == kBad || vf.x == kBad || vf.y == kBad || vf.z == kBad) return;
    i3 a = {blk(vn.x), blk(vn.y), blk(vn.z)}, b = {blk(vf.x), blk(vf.y), blk(vf.z)};
    // The reference's walk along the longest axis, every axis by the error term of
    // its other two: the longest one's (2 M - 1 before each step) is positive each
    // time, so no lane takes another path for its longest axis.
    const int dx = b.x - a.x, dy = b.y - a.y, dz = b.z - a.z;
    const int sx = dx < 0 ? -1 : 1, sy = dy < 0 ? -1 : 1, sz = dz < 0 ? -1 : 1;
    const int ax = abs(dx), ay = abs(dy), az = abs(dz);
    const int steps = max(ax, max(ay, az)), back = steps << 1;
    const int ex = ax << 1, ey = ay << 1, ez = az << 1;
    int e1 = ex - 1, e2 = ey - 1, e3 = ez - 1;
    for (int i = 0;; ++i) {
        emit(a.x, a.y, a.z);
        if (i == steps) break;
        const bool x1 = e1 > 0, y1 = e2 > 0, z1 = e3 > 0;
        a.x += x1 ? sx : 0; e1 += ex - (x1 ? back : 0);
        a.y += y1 ? sy : 0; e2 += ey - (y1 ? back : 0);
        a.z += z1 ? sz : 0; e3 += ez - (z1 ? back : 0);
    }
}

constexpr int kDedup = 1024;  // LDS request set per 16x16 tile (8 KiB)

// Mark an existing block as touched by the current frame (no insertion).
// The mask bit of a block that keyframe re-fusion's band walks created.
constexpr unsigned long long kRefuseFresh = 1ull << 63;

LF_DEV int touch_block(const MapDev &m, int bx, int by, int bz) {
    const unsigned long long key = pack_key(bx, by, bz);
    int slot = compute_hash(bx, by, bz, m.num_buckets);
    for (int i = 0; i < m.num_entries; ++i) {  // find_block, for the slot
        const unsigned long long k = m.keys[slot];
        const int b = m.slot_block[slot];
        if (k == key) {
            if (b < 0) return -1;  // an entry whose block did not fit the pool
            m.slot_flag[slot] = 1;
            return slot;
        }
        if (k == kEmptyKey) return -1;
        if (++slot == m.num_entries) slot = 0;
    }
    return -1;
}

// kInsert: create_blocks_kernel.  !kInsert (de-integration): the same band
// walk only marks the blocks that exist, so the visible list of a frame can be
// rebuilt without allocating.
// 16x16 pixel tile (tx, ty) of the frame.  slot_mask (keyframe re-fusion):
// each block the walk marks also gets `bit` in its hash slot's mask, and
// kRefuseFresh when the walk created it.
// The walks only fill the LDS set and list its keys; then the listed blocks
// go to the hash table side by side, one lane each.  A block's insertion is a
// chain of global accesses, which inside the walks a lane waited for once per
// block it was first to request.  Bound by latency for one frame, by the walks'
// instructions for many: one loop whatever a pixel's longest axis, and a block asked
// for once by neighbours on a row, take 16 frames of 640x480 from 60 to 42 us, 40
// walks of re-fusion from 138 to 111, one frame of 848x480 from 8.6 to 6.5.
struct AllocLds {
    unsigned long long set[kDedup];
    unsigned short list[kDedup];  // positions in the set, in the order of insertion
    unsigned int n;
};
constexpr int kFarTile = 8;
LF_HD int far_tiles(int pixels) { return (pixels + kFarTile - 1) / kFarTile; }
// A depth that the update accepts as an integer of the same order, above 0 (one
// below zero as zero's); 0: a depth it does not.
LF_DEV int far_code(float d, float zmin, float zmax) {
    return isnan(d) || d > zmax || d < zmin ? 0 : __float_as_int(fmaxf(d, 0.0f)) + 1;
}
// The largest far_code of each 8x8-pixel tile of the workgroup's 16x16 pixels into far
// (zero before): a wavefront's four rows of 16 by DPP and permlane swaps, then one
// atomic per tile.
LF_DEV void far_tiles_max(int code, int cols, int rows, int tx, int ty, int *far) {
    code = max(code, __builtin_amdgcn_mov_dpp(code, 0xB1, 0xF, 0xF, false));   // quad_perm 1,0,3,2
    code = max(code, __builtin_amdgcn_mov_dpp(code, 0x4E, 0xF, 0xF, false));   // quad_perm 2,3,0,1
    code = max(code, __builtin_amdgcn_mov_dpp(code, 0x141, 0xF, 0xF, false));  // row_half_mirror
    const auto a = __builtin_amdgcn_permlane16_swap(code, code, false, false);
    code = max((int)a[0], (int)a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(code, code, false, false);
    code = max((int)b[0], (int)b[1]);
    const int t = threadIdx.x, lane = t & 63, x = tx * 2 + (lane >> 3), y = ty * 2 + (t >> 7);
    if ((lane & 7) == 0 && lane < 16 && x < far_tiles(cols) && y < far_tiles(rows) && code > 0)
        atomicMax(&far[y * far_tiles(cols) + x], code);
}

template <bool kInsert, bool kFast, bool kFar = false>
LF_DEV void alloc_wg(const MapDev &m, const float *__restrict__ depth, int cols, int rows,
                     const float *__restrict__ pose24, const lf_intrinsics &K, int tx, int ty, AllocLds &s,
                     unsigned long long *slot_mask = nullptr, unsigned long long bit = 0ull, int *far = nullptr) {
    const int tid = threadIdx.x;
    const int x = tx * 16 + (tid & 15), y = ty * 16 + (tid >> 4);
    const bool inside = x < cols && y < rows;
    // the pixel's depth is in flight while the request set is cleared
    const float z = inside ? depth[(size_t)y * cols + x] : 0.0f;
    for (int i = tid; i < kDedup; i += 256) s.set[i] = kEmptyKey;
    if constexpr (kFar) far_tiles_max(inside ? far_code(z, m.zmin_update, m.zmax_update) : 0, cols, rows, tx, ty, far);
    if (tid == 0) s.n = 0u;
    if (tx == 0 && ty == 0 && tid == 0) {
        m.counters[LF_CNT_VISIBLE] = 0u;
        // one more fusion pass: read by the integration / de-integration that
        // follows this kernel (the seed of the mixed weights' dither).  Atomic, as
        // the 2 n walks of a re-fusion count side by side
        atomicAdd(&m.counters[LF_CNT_FUSE_PASSES], 1u);
    }
    float Twc[12];
#pragma unroll
    for (int i = 0; i < 12; ++i) Twc[i] = pose24[i];
    const auto request = [&](int bx, int by, int bz) {
        bool fresh = false;
        const int slot = kInsert ? insert_block(m, bx, by, bz, &fresh) : touch_block(m, bx, by, bz);
        if (slot_mask && slot >= 0) atomicOr(&slot_mask[slot], bit | (fresh ? kRefuseFresh : 0ull));
    };
    __syncthreads();
    if (inside)
        band_blocks<kFast>(x, y, z, Twc, K, m, [&](int bx, int by, int bz) {
            const unsigned long long key = pack_key(bx, by, bz);
            // Where the pixel to the left asks for the same block at this step, it sees
            // to it: lanes at one address are served in turn.  (row_shr:1; no pixel to
            // the left of a row's first, and none whose walk has ended.)
            const int lo = (int)(unsigned int)key, hi = (int)(unsigned int)(key >> 32);
            const bool left_walks = ((__ballot(1) << 1) >> lane_id() & 1ull) != 0;
            const int left_lo = __builtin_amdgcn_update_dpp(~lo, lo, 0x111, 0xF, 0xF, false),
                      left_hi = __builtin_amdgcn_update_dpp(~hi, hi, 0x111, 0xF, 0xF, false);
            if (left_walks && left_lo == lo && left_hi == hi) return;
            unsigned int h = (unsigned int)(bx + by * 37 + bz * 1369) & (kDedup - 1);
#pragma unroll 1
            for (int probe = 0; probe < kDedup; ++probe) {
                const unsigned long long old = atomicCAS(&s.set[h], kEmptyKey, key);
                if (old == kEmptyKey) {
                    s.list[atomicAdd(&s.n, 1u)] = (unsigned short)h;
                    return;
                }
                if (old == key) return;  // another lane of this tile owns the request
                h = (h + 1) & (kDedup - 1);
            }
            request(bx, by, bz);  // LDS set full: go straight to the table
        });
    __syncthreads();
    for (unsigned int i = tid; i < s.n; i += 256) {
        const unsigned long long key = s.set[s.list[i]];
        request(key_axis(key >> 42), key_axis(key >> 21), key_axis(key));
    }
}

template <bool kInsert, bool kFast = false>
__global__ __launch_bounds__(256) void k_alloc(MapDev m, const float *__restrict__ depth, int cols, int rows,
                                               const float *__restrict__ pose24, lf_intrinsics K) {
    __shared__ AllocLds s;
    alloc_wg<kInsert, kFast>(m, depth, cols, rows, pose24, K, blockIdx.x, blockIdx.y, s);
}

// is_block_visible (depth_fusion.cu:27-47): any of the 8 block corners inside
// the image with z in [zmin, zmax] of the update.  kFast (mixed precision):
// the projection with the hardware reciprocal.
template <bool kFast = false>
LF_DEV bool block_visible(int bx, int by, int bz, const float *Tcw, const lf_intrinsics &K, int cols, int rows,
                          float zmin, float zmax, float scale) {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const float wx = (float)(bx + (c & 1)) * scale, wy = (float)(by + ((c >> 1) & 1)) * scale,
                    wz = (float)(bz + ((c >> 2) & 1)) * scale;
        f3 pt = xform(Tcw, f3{wx, wy, wz});
        float u, v;
        if (kFast) {
            const float iz = __builtin_amdgcn_rcpf(pt.z);
            u = K.fx * pt.x * iz + K.cx;
            v = K.fy * pt.y * iz + K.cy;
        } else if (__builtin_expect(pt.z != 0.0f, 1)) {
            const Recip iz = recip(pt.z);
            u = quotient(K.fx * pt.x, iz) + K.cx;
            v = quotient(K.fy * pt.y, iz) + K.cy;
        } else {
            u = K.fx * pt.x / pt.z + K.cx;
            v = K.fy * pt.y / pt.z + K.cy;
        }
        if (!(u < 0.0f || v < 0.0f || u > (float)(cols - 1) || v > (float)(rows - 1) || pt.z < zmin || pt.z > zmax))
            return true;
    }
    return false;
}

constexpr int kVisThreads = 1024;  // lanes of a k_visible workgroup
constexpr int kVisGrid = 512;      // at most this many workgroups (grid-stride beyond)

// check_visibility_flag_kernel + exclusive scan + copy (depth_fusion.cu:49-93,
// 549-557) over the allocated blocks: touched-this-update, or frustum-visible.
// kGeometric: count_visible_entry (ray_tracing.cu:647-807), frustum-visible
// only, touched flags left alone.  The list is appended with one global atomic
// per workgroup (a wavefront ballot, then the wavefront counts prefixed in
// LDS): same-address atomics serialise, so one per wavefront cost most of the
// kernel.  The list order is unspecified, as with the per-wavefront append.
// Workgroup wg of nwg.
template <bool kGeometric, bool kFast = false>
LF_DEV void visible_wg(const MapDev &m, const float *__restrict__ pose24, const lf_intrinsics &K, int cols, int rows,
                       int wg, int nwg, unsigned int *s_cnt, unsigned int &s_base) {
    float Tcw[12];
#pragma unroll
    for (int i = 0; i < 12; ++i) Tcw[i] = pose24[12 + i];
    const unsigned int stride = nwg * blockDim.x;
    // a lane's first block is loaded beside the number of blocks
    const int4 *bpos = reinterpret_cast<const int4 *>(m.block_pos);
    int4 pos = bpos[min(wg * blockDim.x + threadIdx.x, (unsigned int)m.num_blocks - 1)];
    const unsigned int n = min(m.counters[LF_CNT_ALLOCATED], (unsigned int)m.num_blocks);
    const float scale = 8.0f * m.voxel_size;
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    // the trip count is uniform over the workgroup (its barriers need every lane)
    for (unsigned int b0 = wg * blockDim.x; b0 < n; b0 += stride) {
        const unsigned int b = b0 + threadIdx.x;
        bool vis = false;
        const int4 p = pos;
        pos = bpos[min(b + stride, (unsigned int)m.num_blocks - 1)];
        if (b < n) {
            if (!kGeometric && m.slot_flag[p.w]) {
                vis = true;
                m.slot_flag[p.w] = 0;
            } else {
                vis = block_visible<kFast>(p.x, p.y, p.z, Tcw, K, cols, rows, m.zmin_update, m.zmax_update, scale);
            }
        }
        const unsigned long long ballot = __ballot(vis);
        if (lane == 0) s_cnt[wave] = (unsigned int)__popcll(ballot);
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned int total = 0;
            for (int w = 0; w < kVisThreads / kWave; ++w) {
                const unsigned int c = s_cnt[w];
                s_cnt[w] = total;
                total += c;
            }
            s_base = total ? atomicAdd(&m.counters[LF_CNT_VISIBLE], total) : 0u;
        }
        __syncthreads();
        if (vis) {
            const unsigned int slot = s_base + s_cnt[wave] + __popcll(ballot & ((1ull << lane) - 1ull));
            m.visible[slot] = (int)b;
            reinterpret_cast<int4 *>(m.visible_pos)[slot] = make_int4(p.x, p.y, p.z, (int)b);
        }
        __syncthreads();  // s_cnt and s_base are rewritten by the next iteration
    }
}

template <bool kGeometric = false, bool kFast = false>
__global__ __launch_bounds__(kVisThreads) void k_visible(MapDev m, const float *__restrict__ pose24, lf_intrinsics K,
                                                         int cols, int rows) {
    __shared__ unsigned int s_cnt[kVisThreads / kWave];
    __shared__ unsigned int s_base;
    visible_wg<kGeometric, kFast>(m, pose24, K, cols, rows, blockIdx.x, gridDim.x, s_cnt, s_base);
}

int visible_grid(const lf_map_params *p) {
    return std::min(kVisGrid, std::max(1, (p->num_blocks + kVisThreads - 1) / kVisThreads));
}

// The means' numerators over the new weight, each rounded as by a division; a
// weight outside the range that recip() holds for takes divisions.
template <int kN>
LF_DEV void divide_all(float *n, float w) {
#pragma unroll 1
    for (int k = 0; k < kN; ++k) n[k] /= w;
}
LF_DEV bool recip_holds(float w) { return (w >= 0x1p-60f) & (w <= 0x1p60f); }
template <int kN>
LF_DEV void over_weight(float *n, float w) {
    if (__builtin_expect(recip_holds(w), 1)) {
        const Recip d = recip(w);
#pragma unroll
        for (int k = 0; k < kN; ++k) n[k] = quotient(n[k], d);
    } else {
        divide_all<kN>(n, w);
    }
}

// A pixel's normal (x, y, z of a float4 map whose rows need only be aligned to
// floats) in one load.
struct PackedNormal {
    float x, y, z;
};

// The de-integration of voxel o of a block: its weight w0 (kMixed: of its word),
// sdf code and colours (FP32) as loaded, the frame's observation (sdf in
// truncation units, weight, colour), the stochastic rounding's random bits.
template <bool kColour, bool kMixed>
LF_DEV void take_out_voxel(short *sdf_b, float *w_b, unsigned int *wd_b, unsigned char *c_b, unsigned int o, float w0,
                           unsigned int word, short code, const unsigned char *cold, float sdf, float wt,
                           const unsigned char *cin, unsigned int rnd) {
    if (w0 == 0.0f) return;  // nothing fused here
    const float wr = w0 - wt;
    // mixed: the stored w0 is within one code step (at most 1/16 of it) of the
    // exact sum, so a remainder below that is the rounding of the fused weights
    // and the voxel returns to unseen; a larger one is rounded stochastically, as
    // fusion stores it
    const bool keep = kMixed ? wr > w0 * (1.0f / 16.0f) : wr > 0.0f;
    if (!keep) {
        if constexpr (kMixed) {
            at_byte(sdf_b, 2u * o) = (short)kHalfUnseen;
            at_byte(wd_b, 4u * o) = kColour ? 0u : word & ~0xFFu;  // weight 0; colour cleared with colour fusion
        } else {
            at_byte(sdf_b, 2u * o) = kSdfUnseen;
            at_byte(w_b, 4u * o) = 0.0f;
            if (kColour) {
                at_byte(c_b, o) = 0; at_byte(c_b, o + LF_BLOCK3) = 0; at_byte(c_b, o + 2 * LF_BLOCK3) = 0;
            }
        }
        return;
    }
    const float old = kMixed ? half_bits_to_float((unsigned short)code) : unpack_sdf(code);
    float n[4] = {old * w0 - sdf * wt, 0.0f, 0.0f, 0.0f};
    if (kColour) {
#pragma unroll
        for (int k = 0; k < 3; ++k)
            n[1 + k] = (kMixed ? (float)word_channel(word, k) : (float)cold[k]) * w0 - (float)cin[k] * wt;
    }
    over_weight<kColour ? 4 : 1>(n, wr);
    const float sr = fmaxf(-1.0f, fminf(1.0f, n[0]));
    unsigned int ch[3] = {0u, 0u, 0u};
    if (kColour) {
#pragma unroll
        for (int k = 0; k < 3; ++k) ch[k] = (unsigned int)(int)fmaxf(0.0f, fminf(255.0f, n[1 + k]));
    }
    if constexpr (kMixed) {
        at_byte(sdf_b, 2u * o) = (short)float_to_half_bits(sr);
        at_byte(wd_b, 4u * o) = max(1u, weight_code_sr(wr, rnd)) |
                                (kColour ? word_colour_bits(ch[0], ch[1], ch[2]) : word & ~0xFFu);
    } else {
        at_byte(sdf_b, 2u * o) = pack_sdf(sr);
        at_byte(w_b, 4u * o) = wr;
        if (kColour) {
#pragma unroll
            for (int k = 0; k < 3; ++k) at_byte(c_b, o + k * LF_BLOCK3) = (unsigned char)ch[k];
        }
    }
}

// The 256 weight-code values (weight_value) in LDS: a mixed voxel's weight
// is one LDS read instead of the decode's arithmetic.  Every thread of the
// workgroup calls it.
LF_DEV void fill_weight_table(float *s) {
    for (int i = threadIdx.x; i < 256; i += blockDim.x) s[i] = weight_value((unsigned int)i);
    __syncthreads();
}

// update_map_weighted_kernel (kWeighted, depth_fusion.cu:356-428) and
// update_map_with_colour_kernel (!kWeighted, :288-354).  kPacked (weighted
// only): the pixel's depth, weight and colour come from one 16-byte
// integration sample (DeviceImage frames), whose weight is the same
// expression evaluated when the sample was made; otherwise depth, normal and
// colour are gathered separately.  kMixed: FP16 sdf and 8-bit weight codes,
// and the projection and the weighted means use one reciprocal each instead
// of correctly rounded divisions.
// kTakeOut: de-integration, the inverse of the weighted update for one frame,
// over the same voxels (the selection depends only on depth and pose; the
// projection is correctly rounded in both precisions).  With w the voxel's
// weight and w_f the frame's: w' = w - w_f, sdf' = (sdf w - sdf_f w_f) / w',
// colour likewise; w' <= 0 returns the voxel to unseen.  Exact up to the int16
// sdf and uint8 colour rounding (kMixed: that of the FP16 sdf and the weight
// codes), except where the weight saturated at 255.  Not in the reference
// (deleteBlock, map_struct.cu:327-363, has no callers).
// kTable: the weight codes' values from wtab, an LDS array of 256 floats that
// this function fills (every thread of the workgroup calls it).
// Workgroup wg of nwg (grid-stride over the visible list).
// Bound by the voxels' bytes with packed samples (a 640x480 frame, 5 mm, FP32:
// 238 MB in 53 us; mixed at 848x480, 4 mm: 215 MB in 46 us).  With separate
// planes by the gathers (three a voxel) and the arithmetic: the projection's two
// quotients share one refined reciprocal, the update's four another, a colour and
// a normal are one load each (645x483, 5 mm: 74.6 us with divisions and scalar
// loads, 68.3 now; take-out, a voxel at a time with its loads in sequence before,
// 89.8, now 70.2).  16 mixed maps of 640x480, 5 mm, by both: 2.56 GB, at 4.9 TB/s
// the rate of a large copy, and 421 us of vector instructions: 539 us with the low
// weight codes and the colours' clamps computed for all, 524 now (one map of 848x480,
// 4 mm, 48.3 -> 46.1).
template <bool kWeighted, bool kColour, bool kPacked, bool kMixed, bool kTable = false, bool kTakeOut = false>
LF_DEV void integrate_wg(const MapDev &m, const float *__restrict__ depth, const float *__restrict__ nmap,
                         const unsigned char *__restrict__ rgb, int cols, int rows, const float *__restrict__ pose24,
                         const lf_intrinsics &K, const float4 *__restrict__ samples, int wg, int nwg,
                         float *wtab = nullptr) {
    static_assert(!kPacked || kWeighted, "packed samples carry the weighted update's weight");
    static_assert(!kTakeOut || kWeighted, "only the weighted update is taken out");
    constexpr bool kFast = kMixed && !kTakeOut;  // one hardware reciprocal a projection
    float Tcw[12];
#pragma unroll
    for (int i = 0; i < 12; ++i) Tcw[i] = pose24[12 + i];
    const int nvis = (int)m.counters[LF_CNT_VISIBLE];
    const unsigned int pass = kMixed ? m.counters[LF_CNT_FUSE_PASSES] : 0u;
    // after the loads above: they stay scalar loads ahead of the barrier
    if constexpr (kTable) fill_weight_table(wtab);
    if (!kTakeOut && wg == 0 && threadIdx.x == 0) {
        atomicAdd(&m.counters[LF_CNT_UPDATES], 1u);
        atomicAdd(reinterpret_cast<unsigned long long *>(&m.counters[LF_CNT_VIS_SUM_LO]), (unsigned long long)nvis);
    }
    const float vs = m.voxel_size, trunc = m.truncation, inv_trunc = m.inv_truncation;
    const float zmin = m.zmin_update, zmax = m.zmax_update;
    const int t = threadIdx.x;
    const int lx = t & 7, ly = (t >> 3) & 7, lz0 = t >> 6;
    const float fcols = (float)cols, frows = (float)rows;
    const bool one_pixel = cols * rows == 1;
    // A lane owns voxels t and t + 256 of the block.  Three phases, each
    // issuing both voxels' loads before anything waits on them: the
    // projections and input gathers, then (inside the truncation band) the
    // voxel's weight, sdf and colour together, then the fusion and stores.
    // The block's list entry is the same for every lane (scalar registers,
    // loaded one iteration ahead); voxel and pixel addresses are 32-bit byte
    // offsets from a scalar base.
    // the voxel terms of the stochastic rounding's hash, once per lane
    const unsigned int rand_local[2] = {(unsigned int)t * kRandLocalMul, (unsigned int)(t + 256) * kRandLocalMul};
    const int4 *vpos = reinterpret_cast<const int4 *>(m.visible_pos);  // x, y, z, pool block
    int4 p_next = wg < nvis ? vpos[wg] : make_int4(0, 0, 0, 0);
    for (int i = wg; i < nvis; i += nwg) {
        const int4 p = make_int4(__builtin_amdgcn_readfirstlane(p_next.x), __builtin_amdgcn_readfirstlane(p_next.y),
                                 __builtin_amdgcn_readfirstlane(p_next.z), __builtin_amdgcn_readfirstlane(p_next.w));
        p_next = vpos[min(i + nwg, nvis - 1)];  // unconditional: no wait at a join
        const size_t b = (size_t)p.w;
        short *sdf_b = m.sdf + b * LF_BLOCK3;
        float *w_b = m.weight + b * LF_BLOCK3;
        unsigned int *wd_b = reinterpret_cast<unsigned int *>(m.weight) + b * LF_BLOCK3;  // mixed: voxel words
        unsigned char *c_b = m.rgb + b * (3 * LF_BLOCK3);
        bool ok[2];
        unsigned int pix[2];
        float ptz[2], dist[2], nz[2], wpk[2];
        unsigned int cpk[2];
        f3 pt0 = {0.f, 0.f, 0.f};
        if constexpr (kFast) {
            const float wx = (float)(p.x * 8 + lx) * vs, wy = (float)(p.y * 8 + ly) * vs,
                        wz = (float)(p.z * 8 + lz0) * vs;
            pt0 = xform(Tcw, f3{wx, wy, wz});
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int lz = lz0 + 4 * h;
            f3 pt;
            if constexpr (kFast) {
                // mixed: the second voxel, 4 voxels along z, is one step of the transform's z column
                const float dz = 4.0f * vs;
                pt = h == 0 ? pt0 : f3{pt0.x + Tcw[2] * dz, pt0.y + Tcw[6] * dz, pt0.z + Tcw[10] * dz};
            } else {
                const float wx = (float)(p.x * 8 + lx) * vs, wy = (float)(p.y * 8 + ly) * vs,
                            wz = (float)(p.z * 8 + lz) * vs;
                pt = xform(Tcw, f3{wx, wy, wz});
            }
            // The pixel is (floor(tu), floor(tv)) (__float2int_rd of the
            // rounded projection); it lies in the image exactly when
            // 0 <= tu < cols and 0 <= tv < rows (NaN fails), where the floor
            // is the truncating conversion.
            float tu, tv;
            if constexpr (kFast) {
                const float iz = __builtin_amdgcn_rcpf(pt.z);
                tu = K.fx * pt.x * iz + K.cx + 0.5f;
                tv = K.fy * pt.y * iz + K.cy + 0.5f;
            } else {  // the divisions' floats; a zero z projects nowhere either way
                const Recip iz = recip(pt.z);
                tu = quotient(K.fx * pt.x, iz) + K.cx + 0.5f;
                tv = quotient(K.fy * pt.y, iz) + K.cy + 0.5f;
            }
            // The tests are one mask in FP32 and short-circuited in mixed
            // precision, here and below: the other way round, 645x483 FP32
            // takes 71.0 us, not 68.3, 16 mixed maps 567, not 524.
            if constexpr (kMixed) {
                ok[h] = tu >= 0.0f && tu < fcols && tv >= 0.0f && tv < frows;
                pix[h] = ok[h] ? __umul24((unsigned int)tv, (unsigned int)cols) + (unsigned int)tu : 0u;
            } else {
                ok[h] = (tu >= 0.0f) & (tu < fcols) & (tv >= 0.0f) & (tv < frows);
                const unsigned int at = __umul24((unsigned int)tv, (unsigned int)cols) + (unsigned int)tu;
                pix[h] = ok[h] ? at : 0u;
            }
            ptz[h] = pt.z;
            dist[h] = 0.0f; nz[h] = 0.0f; wpk[h] = 0.0f; cpk[h] = 0u;
        }
        // The gathers and voxel loads below are unconditional, so that both
        // voxels' loads issue before the first wait: a lane with nothing to
        // load reads pixel 0, or voxel 0 of its block, and its values are
        // never used.  Mixed precision reads every voxel's sdf and word in
        // the same round as the gathers (one memory round trip before the
        // fusion instead of two, for the bytes of the voxels the band leaves
        // out).
        unsigned int word[2], vo[2];
        short sp[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            vo[h] = vgpr_offset((unsigned int)(t + 256 * h));
            if constexpr (kMixed) {
                word[h] = at_byte(wd_b, 4u * vo[h]);  // weight code and colour together
                sp[h] = at_byte(sdf_b, 2u * vo[h]);
            }
        }
        float nx[2] = {0.0f, 0.0f};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (kPacked) {
                const float4 smp = at_byte(samples, vgpr_offset(16u * pix[h]));
                dist[h] = smp.x;  // NaN also when the normal is invalid
                wpk[h] = smp.y;
                cpk[h] = __float_as_uint(smp.z);
            } else {
                dist[h] = at_byte(depth, 4u * pix[h]);
                if (kWeighted) {
                    const PackedNormal n = at_byte(reinterpret_cast<const PackedNormal *>(nmap), 16u * pix[h]);
                    nx[h] = n.x;
                    nz[h] = n.z;
                }
                if (kColour) cpk[h] = rgb_at(rgb, pix[h], one_pixel);
            }
        }
        float sdf[2], wraw[2];
        unsigned char cold[2][3];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float d = dist[h];
            bool in = ok[h];
            if constexpr (kMixed) {
                if (kPacked) in = in && !(isnan(d) || d > zmax || d < zmin);
                else if (kWeighted) in = in && !(isnan(d) || isnan(nx[h]) || d > zmax || d < zmin);
                else in = in && !(isnan(d) || (double)d < 1e-2 || d > zmax || d < zmin);
                sdf[h] = d - ptz[h];
                in = in && !(sdf[h] < -trunc);
            } else {
                sdf[h] = d - ptz[h];
                in = in & !(d > zmax) & !(d < zmin) & (sdf[h] >= -trunc);  // a NaN depth fails the last
                if (!kPacked && kWeighted) in = in & !isnan(nx[h]);
                if (!kWeighted) in = in & !((double)d < 1e-2);
            }
            ok[h] = in;
            if constexpr (!kMixed) {
                const unsigned int o = in ? vo[h] : 0u;
                wraw[h] = at_byte(w_b, 4u * o);
                if (kColour) {
                    cold[h][0] = at_byte(c_b, o);
                    cold[h][1] = at_byte(c_b, o + LF_BLOCK3);
                    cold[h][2] = at_byte(c_b, o + 2 * LF_BLOCK3);
                }
                sp[h] = at_byte(sdf_b, 2u * o);
            }
        }
        float wp[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
            wp[h] = kMixed ? (kTable ? wtab[word_code(word[h])] : weight_value(word_code(word[h]))) : wraw[h];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (!ok[h]) continue;
            const float d = dist[h];
            const float sdf_h = fminf(1.0f, sdf[h] * inv_trunc);
            const unsigned int o = vo[h];
            const float wt = kPacked ? wpk[h] : kWeighted ? fabsf(sinf(nz[h])) / (d * d) : 1.0f / (d * d);
            unsigned char cin[3];
            if (kColour) {
#pragma unroll
                for (int k = 0; k < 3; ++k) cin[k] = (unsigned char)(cpk[h] >> (8 * k));
            }
            if constexpr (kTakeOut) {
                take_out_voxel<kColour, kMixed>(sdf_b, w_b, wd_b, c_b, o, wp[h], word[h], sp[h], cold[h], sdf_h, wt,
                                                cin, voxel_rand_mixed(p.x, p.y, p.z, rand_local[h], pass));
                continue;
            }
            if constexpr (kMixed) {
                unsigned short *sdf16 = reinterpret_cast<unsigned short *>(sdf_b);
                // the stored weight is rounded stochastically (unbiased running sums)
                const unsigned int rnd = voxel_rand_mixed(p.x, p.y, p.z, rand_local[h], pass);
                // without colour fusion the word's colour bits are kept
                unsigned int colour = word[h] & ~0xFFu;
                if (wp[h] == 0.0f) {
                    // a first observation with a positive weight is seen, as in
                    // the reference (the smallest code stands for weights below
                    // it); a zero weight leaves the voxel unseen
                    const unsigned int code =
                        wt > 0.0f ? max(1u, weight_code_sr_in_range(fminf(wt, 255.0f), rnd)) : 0u;
                    at_byte(sdf16, vgpr_offset(2u * o)) = code == 0u ? kHalfUnseen : float_to_half_bits(sdf_h);
                    if (kColour) colour = word_colour_bits(cin[0], cin[1], cin[2]);
                    at_byte(wd_b, vgpr_offset(4u * o)) = code | colour;
                    continue;
                }
                const float wn = wp[h] + wt, inv = __builtin_amdgcn_rcpf(wn);
                const float spf = half_bits_to_float((unsigned short)sp[h]);
                at_byte(sdf16, vgpr_offset(2u * o)) = float_to_half_bits((spf * wp[h] + sdf_h * wt) * inv);
                unsigned int code = weight_code_sr_normal(fminf(wn, 255.0f), rnd);
                float mc[3];
                if (kColour) {
#pragma unroll
                    for (int k = 0; k < 3; ++k)
                        mc[k] = ((float)word_channel(word[h], k) * wp[h] + (float)cin[k] * wt) * inv;
                    colour = word_colour_of(mc[0], mc[1], mc[2]);
                }
                // Few wavefronts hold a weight below 2^-6 or one that makes the means NaN (not
                // finite, or past 2^60 here): their codes and clamps, with one test for both
                // (a clamp for all: 526.5 us for the 16 maps' 523.4).
                if (__builtin_expect(__any(__float_as_uint(wn) - (121u << 23) > (187u - 121u) << 23), 0)) {
                    code = weight_code_sr(fminf(wn, 255.0f), rnd);
                    if (kColour) colour = word_colour_of(fminf(mc[0], 255.0f), fminf(mc[1], 255.0f), fminf(mc[2], 255.0f));
                }
                at_byte(wd_b, vgpr_offset(4u * o)) = code | colour;
                continue;
            }
            if (wp[h] == 0.0f) {
                // weight stays 0 only when wt is 0: keep the voxel's sdf code unseen
                at_byte(sdf_b, 2u * o) = wt == 0.0f ? kSdfUnseen : pack_sdf(sdf_h);
                at_byte(w_b, 4u * o) = wt > 255.0f ? 255.0f : wt;
                if (kColour) {
                    at_byte(c_b, o) = cin[0]; at_byte(c_b, o + LF_BLOCK3) = cin[1];
                    at_byte(c_b, o + 2 * LF_BLOCK3) = cin[2];
                }
                continue;
            }
            const float spf = unpack_sdf(sp[h]);
            const float wn = wp[h] + wt;
            float n[4] = {spf * wp[h] + sdf_h * wt, 0.0f, 0.0f, 0.0f};
            if (kColour) {
#pragma unroll
                for (int k = 0; k < 3; ++k) n[1 + k] = (float)cold[h][k] * wp[h] + (float)cin[k] * wt;
            }
            over_weight<kColour ? 4 : 1>(n, wn);
            at_byte(sdf_b, 2u * o) = pack_sdf(n[0]);
            at_byte(w_b, 4u * o) = wn > 255.0f ? 255.0f : wn;
            if (kColour) {
#pragma unroll
                for (int k = 0; k < 3; ++k) at_byte(c_b, o + k * LF_BLOCK3) = (unsigned char)(int)n[1 + k];
            }
        }
    }
}

template <bool kWeighted, bool kColour, bool kPacked = false, bool kMixed = false>
__global__ __launch_bounds__(256) void k_integrate(MapDev m, const float *__restrict__ depth,
                                                   const float *__restrict__ nmap,
                                                   const unsigned char *__restrict__ rgb, int cols, int rows,
                                                   const float *__restrict__ pose24, lf_intrinsics K,
                                                   const float4 *__restrict__ samples = nullptr) {
    __shared__ float s_wv[kMixed ? 256 : 1];
    integrate_wg<kWeighted, kColour, kPacked, kMixed, kMixed>(m, depth, nmap, rgb, cols, rows, pose24, K, samples,
                                                              blockIdx.x, gridDim.x, s_wv);
}

// One map's weighted update from a frame's packed samples within a batch
// (each a 2-D launch whose y index is the map): the arguments of the three
// kernels, and each map's grids.
struct FuseJob {
    MapDev m;
    const float *depth;
    const float4 *samples;
    const unsigned char *rgb;  // null: no colour
    const float *pose24;
    lf_intrinsics K;
    int cols, rows, tiles_x, tiles_y, vis_grid;
};

template <bool kFast>
__global__ __launch_bounds__(256) void k_alloc_batch(const FuseJob *__restrict__ jobs) {
    __shared__ AllocLds s;
    const FuseJob &j = jobs[blockIdx.y];
    const int t = blockIdx.x;
    if (t >= j.tiles_x * j.tiles_y) return;
    alloc_wg<true, kFast>(global_dev(j.m), global_ptr(j.depth), j.cols, j.rows, global_ptr(j.pose24), j.K,
                          t % j.tiles_x, t / j.tiles_x, s);
}

template <bool kFast>
__global__ __launch_bounds__(kVisThreads) void k_visible_batch(const FuseJob *__restrict__ jobs) {
    __shared__ unsigned int s_cnt[kVisThreads / kWave];
    __shared__ unsigned int s_base;
    const FuseJob &j = jobs[blockIdx.y];
    if ((int)blockIdx.x >= j.vis_grid) return;
    visible_wg<false, kFast>(global_dev(j.m), global_ptr(j.pose24), j.K, j.cols, j.rows, blockIdx.x, j.vis_grid, s_cnt,
                      s_base);
}

template <bool kMixed>
__global__ __launch_bounds__(256) void k_integrate_batch(const FuseJob *__restrict__ jobs) {
    __shared__ float s_wv[256];
    const FuseJob &j = jobs[blockIdx.y];
    if (j.tiles_x == 0) return;  // a map without an update this step (the whole workgroup)
    const MapDev m = global_dev(j.m);
    const float *depth = global_ptr(j.depth), *pose24 = global_ptr(j.pose24);
    const float4 *samples = global_ptr(j.samples);
    const unsigned char *rgb = global_ptr(j.rgb);
    if (rgb)
        integrate_wg<true, true, true, kMixed, kMixed>(m, depth, nullptr, rgb, j.cols, j.rows, pose24, j.K, samples,
                                                       blockIdx.x, gridDim.x, s_wv);
    else
        integrate_wg<true, false, true, kMixed, kMixed>(m, depth, nullptr, rgb, j.cols, j.rows, pose24, j.K, samples,
                                                        blockIdx.x, gridDim.x, s_wv);
}

template <bool kColour, bool kPacked, bool kMixed = false>
__global__ __launch_bounds__(256) void k_deintegrate(MapDev m, const float *__restrict__ depth,
                                                     const float *__restrict__ nmap,
                                                     const unsigned char *__restrict__ rgb, int cols, int rows,
                                                     const float *__restrict__ pose24, lf_intrinsics K,
                                                     const float4 *__restrict__ samples) {
    __shared__ float s_wv[kMixed ? 256 : 1];
    integrate_wg<true, kColour, kPacked, kMixed, kMixed, true>(m, depth, nmap, rgb, cols, rows, pose24, K, samples,
                                                               blockIdx.x, gridDim.x, s_wv);
}

// ------------------------------------------------------------ keyframe re-fusion
//
// n keyframes (each a frame's raw depth and packed integration samples, all of
// one size and intrinsics) leave the map at their old poses and are fused at
// their new poses in one pass: block allocation for every keyframe at its new
// pose (one launch), the union of the blocks any old or new pose sees (one
// launch), then one lane per voxel replays, in registers, the de-integration
// of keyframes 0..n-1 at their old poses followed by their weighted update at
// the new poses, in that order, and stores once.  Each step follows
// k_deintegrate / the weighted update (depth_fusion.cu:356-428) for that
// voxel, so the result is that of the 2n launches in sequence except that the
// voxel is not re-quantised between the steps.  A keyframe's step touches the
// blocks its own launches would have listed: those its pose sees
// (is_block_visible, depth_fusion.cu:27-47) and those the band walk of its
// depth at that pose marks (create_blocks_kernel, depth_fusion.cu:121-228;
// the old poses' walks only mark blocks that exist), recorded per hash slot
// as one bit per keyframe and pose.  A block this call creates did not exist
// for the de-integrations, nor for the updates before that of the first
// keyframe whose walk reaches it (in sequence it would be allocated there).
constexpr int kMaxRefuse = LF_REFUSE_MAX_KEYFRAMES;  // 2 poses each: one wavefront's lanes
static_assert(2 * kMaxRefuse < 64, "a wavefront tests every pose of a block; bit 63 marks new blocks");

struct RefuseArgs {
    MapDev m;
    unsigned long long *slot_mask;  // per hash slot: bit k old pose k, bit n + k new pose k
    unsigned long long *list_mask;  // per visible-list entry: the poses whose steps it takes, the same bits
    int *tile_far;                  // per keyframe and kFarTile^2 pixels: far_code of the largest depth in range
    const float *depth[kMaxRefuse];
    const float4 *samples[kMaxRefuse];
    const float *old24[kMaxRefuse];
    const float *new24[kMaxRefuse];
    int n, cols, rows;
    lf_intrinsics K;
};

__global__ void k_fill_u64(unsigned long long *p, size_t n) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = 0ull;
}

// Row y < n of the grid: keyframe y's band walk at its old pose (existing
// blocks only) and its tile_far; row n + k: keyframe k's at its new pose, allocating.
template <bool kFast>
__global__ __launch_bounds__(256) void k_refuse_alloc(RefuseArgs a) {
    __shared__ AllocLds s;
    const int tiles_x = (a.cols + 15) / 16;
    const int y = blockIdx.y, t = blockIdx.x;
    if (y < a.n)
        alloc_wg<false, kFast, true>(a.m, a.depth[y], a.cols, a.rows, a.old24[y], a.K, t % tiles_x, t / tiles_x, s,
                                     a.slot_mask, 1ull << y,
                                     a.tile_far + (size_t)y * far_tiles(a.cols) * far_tiles(a.rows));
    else
        alloc_wg<true, kFast>(a.m, a.depth[y - a.n], a.cols, a.rows, a.new24[y - a.n], a.K, t % tiles_x,
                              t / tiles_x, s, a.slot_mask, 1ull << y);
}

// Pose j of the 2n (j < n: keyframe j's old pose, else keyframe j - n's new
// pose) as a float T_cw.
LF_DEV const float *refuse_pose(const RefuseArgs &a, int j) {
    return (j < a.n ? a.old24[j] : a.new24[j - a.n]) + 12;
}

// The largest of a wavefront's 64 values, in every lane.
LF_DEV int wave_max(int v) {
    v = max(v, __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, false));   // quad_perm 1,0,3,2
    v = max(v, __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, false));   // quad_perm 2,3,0,1
    v = max(v, __builtin_amdgcn_mov_dpp(v, 0x141, 0xF, 0xF, false));  // row_half_mirror
    v = max(v, __builtin_amdgcn_mov_dpp(v, 0x128, 0xF, 0xF, false));  // row_ror:8
    const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = max((int)a[0], (int)a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return max((int)b[0], (int)b[1]);
}

// Whether a pose surely sees no corner of the block around the camera point c
// (every corner within r of it, the rounding of c and of block_visible's
// projections included): behind or beyond the update range, or outside one of the
// image's four planes.
LF_DEV bool surely_unseen(f3 c, float r, const lf_intrinsics &K, int cols, int rows, float zmin, float zmax) {
    if (c.z + r < zmin || c.z - r > zmax) return true;
    if (!(c.z - r > 0.0f)) return false;  // a corner may lie behind the camera: its projection flips
    // u < 0 <=> fx x + cx z < 0; u > cols - 1 <=> fx x + (cx - cols + 1) z > 0
    const float gu = K.fx * c.x + K.cx * c.z, hu = gu - (float)(cols - 1) * c.z;
    const float gv = K.fy * c.y + K.cy * c.z, hv = gv - (float)(rows - 1) * c.z;
    const float ru = r * (fabsf(K.fx) + fabsf(K.cx) + (float)cols), rv = r * (fabsf(K.fy) + fabsf(K.cy) + (float)rows);
    return gu < -ru || hu > ru || gv < -rv || hv > rv;
}

// What a pose T_cw makes of a block: radius, around its centre, of its corners; half and
// shift, the camera-aligned box around its voxels (half sizes, centre relative to the
// block's).  Each with a hundredth of a block to spare, and for any linear part, not
// rotations alone.
// A block at P (its largest coordinate) is transformed with a rounding of at most 2^-20 M,
// M = row sum of |T_cw| times P plus the translation: 14 roundings of 2^-24 for a point and
// the centre.  The same again covers block_visible's projections: a slack of
// scale P + offset.
struct RefuseBox {
    f3 half, shift;
};
struct RefuseSlack {
    float radius, scale, offset;
};
LF_DEV RefuseBox refuse_box(const float *Tcw, float vs, RefuseSlack &s) {
    RefuseBox b;
    float *h = &b.half.x, *c = &b.shift.x;
    float rows = 0.0f, offset = 0.0f, gram = 0.0f;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const float x = Tcw[4 * i], y = Tcw[4 * i + 1], z = Tcw[4 * i + 2], row = fabsf(x) + fabsf(y) + fabsf(z);
        h[i] = 3.5f * vs * row + 0.08f * vs;
        c[i] = -0.5f * vs * (x + y + z);  // voxels 0..7 around 3.5
        rows = fmaxf(rows, row);
        offset = fmaxf(offset, fabsf(Tcw[4 * i + 3]));
        float sum = 0.0f;  // row i of T^t T, whose largest bounds the square of T's norm (1 for a rotation)
#pragma unroll
        for (int j = 0; j < 3; ++j) sum += fabsf(Tcw[i] * Tcw[j] + Tcw[4 + i] * Tcw[4 + j] + Tcw[8 + i] * Tcw[8 + j]);
        gram = fmaxf(gram, sum);
    }
    // half a block's diagonal is 0.8660 of its side
    s.radius = (8.0f * vs) * fmaf(0.867f, __builtin_amdgcn_sqrtf(gram), 0.008f);
    s.scale = 0x1p-19f * rows;
    s.offset = 0x1p-19f * offset;
    return b;
}

// Whether keyframe k changes no voxel of the block whose box at this pose is
// c +- half (their rounding included): every voxel that projects into the image lies more
// than the truncation behind the largest depth of the tiles around it (or the tiles hold
// no depth).
// The box's pixels are widened by one for the rounding of the voxels' projections.
LF_DEV bool surely_behind(const RefuseArgs &a, int k, f3 c, f3 half) {
    const float zn = c.z - half.z, zf = c.z + half.z;
    if (!(zn > 0.0f) || !(a.K.fx > 0.0f) || !(a.K.fy > 0.0f)) return false;
    const float in = __builtin_amdgcn_rcpf(zn), fn = __builtin_amdgcn_rcpf(zf);
    const float x0 = c.x - half.x, x1 = c.x + half.x, y0 = c.y - half.y, y1 = c.y + half.y;
    const float u0 = a.K.fx * x0 * (x0 < 0.0f ? in : fn) + a.K.cx - 0.5f,
                u1 = a.K.fx * x1 * (x1 > 0.0f ? in : fn) + a.K.cx + 1.5f,
                v0 = a.K.fy * y0 * (y0 < 0.0f ? in : fn) + a.K.cy - 0.5f,
                v1 = a.K.fy * y1 * (y1 > 0.0f ? in : fn) + a.K.cy + 1.5f;
    if (!(u1 - u0 < 4.0f * kFarTile) || !(v1 - v0 < 4.0f * kFarTile)) return false;  // at most 5x5 tiles; NaN
    const int w = far_tiles(a.cols), h = far_tiles(a.rows);
    const int tx0 = (int)fmaxf(u0, 0.0f) / kFarTile, tx1 = (int)fminf(u1, (float)(a.cols - 1)) / kFarTile;
    const int ty0 = (int)fmaxf(v0, 0.0f) / kFarTile, ty1 = (int)fminf(v1, (float)(a.rows - 1)) / kFarTile;
    const int *far = a.tile_far + (size_t)k * w * h;
    int most = 0;
    if (u1 >= 0.0f && v1 >= 0.0f)
        for (int y = ty0; y <= ty1; y += 3)  // nine tiles' loads in flight, the last row and column repeated
            for (int x = tx0; x <= tx1; x += 3)
#pragma unroll
                for (int i = 0; i < 9; ++i) most = max(most, far[min(y + i / 3, ty1) * w + min(x + i % 3, tx1)]);
    return most == 0 || __int_as_float(most - 1) - zn < -a.m.truncation * 1.0001f;
}

// The visible list becomes every allocated block that a keyframe's old or new
// pose sees or whose slot the band walks marked (the slot flags are cleared),
// each with the mask of the poses whose steps it takes, less those whose depths all
// lie in front of the block.  Four lanes test a block, every fourth pose each, and
// only the poses that a bounding sphere leaves open corner by corner.  40 poses of
// 165k blocks: 104 us with one lane per block and no sphere; 39 without the depths'
// test, 54 with it, which takes 160 us off k_refuse (tiles of 4 pixels, as good a
// test: 70).  Bound by the latency of a lane's chain of poses: 60 -> 44 us (under the
// profiler) with nine tiles' loads in flight and three workgroups of 512 lanes on a CU
// for one of 1024 (77 VGPRs; 57 at 64 VGPRs and 1024 lanes, 50 with 256 lanes).
constexpr int kRefuseVisThreads = 512;
template <bool kFast>
__global__ __launch_bounds__(kRefuseVisThreads, 6) void k_refuse_visible(RefuseArgs a) {
    __shared__ unsigned int s_cnt[kRefuseVisThreads / kWave];
    __shared__ unsigned int s_base;
    __shared__ float s_pose[2 * kMaxRefuse][12];
    __shared__ RefuseBox s_box[2 * kMaxRefuse];
    __shared__ int s_most[3];  // the largest radius, slack scale and offset of all poses, as bits
    const MapDev &m = a.m;
    for (int i = threadIdx.x; i < 2 * a.n * 12; i += kRefuseVisThreads)
        s_pose[i / 12][i % 12] = refuse_pose(a, i / 12)[i % 12];
    __syncthreads();
    if (threadIdx.x < kWave) {  // a lane a pose
        const int i = threadIdx.x;
        RefuseSlack s = {0.0f, 0.0f, 0.0f};
        if (i < 2 * a.n) s_box[i] = refuse_box(s_pose[i], m.voxel_size, s);
        // (the bits of a NaN, from a pose that is not finite, are the largest: no test below says unseen then)
        int most[3] = {__float_as_int(s.radius), __float_as_int(s.scale), __float_as_int(s.offset)};
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            most[k] = wave_max(most[k] & 0x7FFFFFFF);
            if (i == 0) s_most[k] = most[k];
        }
    }
    __syncthreads();
    // One bound for all poses, the same in every lane.  (20 keyframes: 39.0 us without the
    // slack, 40.1 with it; a radius and slack per pose 45, the maxima by LDS atomics 59.)
    const auto uniform = [&](int i) { return __int_as_float(__builtin_amdgcn_readfirstlane(s_most[i])); };
    const RefuseSlack most = {uniform(0), uniform(1), uniform(2)};
    const unsigned int nb = min(m.counters[LF_CNT_ALLOCATED], (unsigned int)m.num_blocks);
    const float scale = 8.0f * m.voxel_size;
    constexpr unsigned int kPerWg = kRefuseVisThreads / 4;
    const unsigned int stride = gridDim.x * kPerWg;
    const int lane = lane_id(), wave = threadIdx.x / kWave, sub = threadIdx.x & 3;
    const unsigned long long all = (1ull << a.n) - 1ull;
    for (unsigned int b0 = blockIdx.x * kPerWg; b0 < nb; b0 += stride) {
        const unsigned int b = b0 + threadIdx.x / 4;
        bool vis = false;
        int4 p = make_int4(0, 0, 0, 0);
        unsigned long long steps = 0ull, seen = 0ull, idle = 0ull, marks = 0ull;
        bool flagged = false;
        if (b < nb) {
            p = reinterpret_cast<const int4 *>(m.block_pos)[b];
            marks = a.slot_mask[p.w];
            flagged = m.slot_flag[p.w] != 0;
            const f3 centre = {((float)p.x + 0.5f) * scale, ((float)p.y + 0.5f) * scale, ((float)p.z + 0.5f) * scale};
            const float P = fmaxf(fmaxf(fabsf(centre.x), fabsf(centre.y)), fabsf(centre.z)) + scale;
            const float e = fmaf(most.scale, P, most.offset);
            unsigned int open = 0u;  // bit i: pose sub + 4 i
            for (int i = 0, j = sub; j < 2 * a.n; ++i, j += 4)
                if (!surely_unseen(xform(s_pose[j], centre), most.radius + e, a.K, a.cols, a.rows, m.zmin_update,
                                   m.zmax_update))
                    open |= 1u << i;
            for (; open; open &= open - 1u) {
                const int j = sub + 4 * __builtin_ctz(open);
                if (!block_visible<kFast>(p.x, p.y, p.z, s_pose[j], a.K, a.cols, a.rows, m.zmin_update, m.zmax_update,
                                          scale))
                    continue;
                seen |= 1ull << j;
                const f3 c = add(xform(s_pose[j], centre), s_box[j].shift);
                if (surely_behind(a, j < a.n ? j : j - a.n, c, add(s_box[j].half, f3{e, e, e})))
                    idle |= 1ull << j;
            }
        }
        seen |= __shfl_xor(seen, 1);
        seen |= __shfl_xor(seen, 2);
        idle |= __shfl_xor(idle, 1);
        idle |= __shfl_xor(idle, 2);
        if (b < nb && sub == 0) {
            if (flagged) m.slot_flag[p.w] = 0;
            seen |= marks & ~kRefuseFresh;
            vis = flagged || marks != 0ull || seen != 0ull;
            unsigned long long old_mask = seen & all, new_mask = (seen >> a.n) & all;
            if (marks & kRefuseFresh) {
                // created here: by the first keyframe whose new-pose walk reached it
                const unsigned long long walks = (marks >> a.n) & all;
                old_mask = 0ull;
                new_mask &= ~((walks & (0ull - walks)) - 1ull);
            }
            steps = (old_mask | new_mask << a.n) & ~idle;
        }
        const unsigned long long ballot = __ballot(vis);
        if (lane == 0) s_cnt[wave] = (unsigned int)__popcll(ballot);
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned int total = 0;
            for (int w = 0; w < kRefuseVisThreads / kWave; ++w) {
                const unsigned int c = s_cnt[w];
                s_cnt[w] = total;
                total += c;
            }
            s_base = total ? atomicAdd(&m.counters[LF_CNT_VISIBLE], total) : 0u;
        }
        __syncthreads();
        if (vis) {
            const unsigned int slot = s_base + s_cnt[wave] + __popcll(ballot & ((1ull << lane) - 1ull));
            m.visible[slot] = (int)b;
            reinterpret_cast<int4 *>(m.visible_pos)[slot] = make_int4(p.x, p.y, p.z, (int)b);
            a.list_mask[slot] = steps;
        }
        __syncthreads();
    }
}

// A keyframe's observation of a voxel before its sample has arrived: its depth in
// the camera, infinite where it does not project into the image, and its pixel.
struct RefuseProj {
    float z;
    unsigned int pix;
};
// kFast: the hardware reciprocal projection of the mixed-precision update.
template <bool kFast>
LF_DEV RefuseProj refuse_project(const RefuseArgs &a, const float *Tcw, float wx, float wy, float wz) {
    const f3 pt = xform(Tcw, f3{wx, wy, wz});
    float tu, tv;
    if (kFast) {
        const float iz = __builtin_amdgcn_rcpf(pt.z);
        tu = a.K.fx * pt.x * iz + a.K.cx + 0.5f;
        tv = a.K.fy * pt.y * iz + a.K.cy + 0.5f;
    } else {  // a zero z projects nowhere either way
        const Recip iz = recip(pt.z);
        tu = quotient(a.K.fx * pt.x, iz) + a.K.cx + 0.5f;
        tv = quotient(a.K.fy * pt.y, iz) + a.K.cy + 0.5f;
    }
    // the pixel (floor(tu), floor(tv)), in the image exactly when 0 <= tu < cols
    // and 0 <= tv < rows (NaN fails), where the floor is the truncating conversion
    const bool in = (tu >= 0.0f) & (tu < (float)a.cols) & (tv >= 0.0f) & (tv < (float)a.rows);
    const unsigned int pix = __umul24((unsigned int)(int)tv, (unsigned int)a.cols) + (unsigned int)(int)tu;
    return {in ? pt.z : __builtin_inff(), in ? pix : 0u};
}

// A voxel's running mean (sdf, colour) and weight.
struct RefuseVoxel {
    float w, sdf, col[3];
    bool changed;
};

// take_out_voxel's arithmetic on a running mean.
template <bool kColour, bool kMixed>
LF_DEV void refuse_take_out(RefuseVoxel &v, float s, float wt, unsigned int rgb) {
    v.changed = true;
    const float wr = v.w - wt;
    const bool keep = kMixed ? wr > v.w * (1.0f / 16.0f) : wr > 0.0f;
    if (!keep) {
        v.w = 0.0f;
        v.sdf = 0.0f;
        if (kColour) v.col[0] = v.col[1] = v.col[2] = 0.0f;
        return;
    }
    float n[4] = {v.sdf * v.w - s * wt, 0.0f, 0.0f, 0.0f};
    if (kColour) {
#pragma unroll
        for (int q = 0; q < 3; ++q) n[1 + q] = v.col[q] * v.w - (float)((rgb >> (8 * q)) & 0xFFu) * wt;
    }
    divide_all<kColour ? 4 : 1>(n, wr);
    v.sdf = fmaxf(-1.0f, fminf(1.0f, n[0]));
    if (kColour) {
#pragma unroll
        for (int q = 0; q < 3; ++q) v.col[q] = fmaxf(0.0f, fminf(255.0f, n[1 + q]));
    }
    v.w = wr;
}

// The weighted update's.
template <bool kColour>
LF_DEV void refuse_put_in(RefuseVoxel &v, float s, float wt, unsigned int rgb) {
    v.changed = true;
    if (v.w == 0.0f) {
        v.sdf = s;
        v.w = fminf(wt, 255.0f);
        if (kColour) {
#pragma unroll
            for (int q = 0; q < 3; ++q) v.col[q] = (float)((rgb >> (8 * q)) & 0xFFu);
        }
        return;
    }
    const float wn = v.w + wt;
    float n[4] = {v.sdf * v.w + s * wt, 0.0f, 0.0f, 0.0f};
    if (kColour) {
#pragma unroll
        for (int q = 0; q < 3; ++q) n[1 + q] = v.col[q] * v.w + (float)((rgb >> (8 * q)) & 0xFFu) * wt;
    }
    divide_all<kColour ? 4 : 1>(n, wn);
    v.sdf = n[0];
    if (kColour) {
#pragma unroll
        for (int q = 0; q < 3; ++q) v.col[q] = n[1 + q];
    }
    v.w = fminf(wn, 255.0f);
}

// One step of a voxel, de-integration or update (the same for a whole wavefront):
// with the frame's weight signed, both are the mean of the two over w + ws, the
// de-integration's clamped.  A first observation, a voxel that returns to unseen and
// a weight outside recip()'s range take the functions above.
template <bool kColour, bool kMixed>
LF_DEV void refuse_step(RefuseVoxel &v, float s, float wt, unsigned int rgb, bool put_in) {
    const float ws = put_in ? wt : -wt, wn = v.w + ws;
    const bool plain = (put_in ? v.w : wn) > (kMixed && !put_in ? v.w * (1.0f / 16.0f) : 0.0f);
    if (plain & recip_holds(wn)) {
        const Recip d = recip(wn);
        v.changed = true;
        v.sdf = quotient(v.sdf * v.w + s * ws, d);
        if (kColour) {
#pragma unroll
            for (int q = 0; q < 3; ++q)
                v.col[q] = quotient(v.col[q] * v.w + (float)((rgb >> (8 * q)) & 0xFFu) * ws, d);
        }
        if (!put_in) {
            v.sdf = __builtin_amdgcn_fmed3f(v.sdf, -1.0f, 1.0f);
            if (kColour) {
#pragma unroll
                for (int q = 0; q < 3; ++q) v.col[q] = __builtin_amdgcn_fmed3f(v.col[q], 0.0f, 255.0f);
            }
        }
        v.w = fminf(wn, 255.0f);
    } else if (put_in) {
        refuse_put_in<kColour>(v, s, wt, rgb);
    } else if (v.w != 0.0f) {
        refuse_take_out<kColour, kMixed>(v, s, wt, rgb);
    }
}

// One lane per voxel (two voxels per lane, 256 lanes per block) of the visible
// list: the steps of its mask in order, de-integrations (bits below n) first.
// kMixed: FP16 sdf and the packed weight-code / colour word, the weights
// rounded stochastically once at the end (as the update stores them).
// Each step gathers 16 bytes per voxel: both voxels' samples of the next step
// are loaded while the present one is applied, and the poses are in LDS.
// Bound by its vector instructions (the arithmetic of a projection and of four
// weighted means a voxel and step).  20 keyframes of 640x480 on 165k blocks (FP32,
// 4 mm): 1797 us at one voxel and one load after the other, 966 with divisions'
// branches for either direction, 775 with the steps that change nothing left
// out, 762 now with the clamps only where they can act.
// 64 VGPRs keep 8 waves a SIMD (66: 1018 us where 64 took 934).
template <bool kColour, bool kMixed>
__global__ __launch_bounds__(256, 8) void k_refuse(RefuseArgs a) {
    __shared__ float s_pose[2 * kMaxRefuse][12];
    const MapDev &m = a.m;
    const int t = threadIdx.x;
    for (int i = t; i < 2 * a.n * 12; i += 256) s_pose[i / 12][i % 12] = refuse_pose(a, i / 12)[i % 12];
    __syncthreads();
    const int nvis = (int)m.counters[LF_CNT_VISIBLE];
    const unsigned int pass = kMixed ? m.counters[LF_CNT_FUSE_PASSES] : 0u;
    const float vs = m.voxel_size, zmin = m.zmin_update, zmax = m.zmax_update;
    const int lx = t & 7, ly = (t >> 3) & 7, lz0 = t >> 6;
    unsigned short *sdf16 = reinterpret_cast<unsigned short *>(m.sdf);
    unsigned int *wd = reinterpret_cast<unsigned int *>(m.weight);
    for (int i = blockIdx.x; i < nvis; i += gridDim.x) {
        const int4 p = reinterpret_cast<const int4 *>(m.visible_pos)[i];
        const unsigned long long mask = a.list_mask[i];
        // the mask in scalar registers: the steps are the same for every lane
        const unsigned int lo = (unsigned int)__builtin_amdgcn_readfirstlane((int)mask),
                           hi = (unsigned int)__builtin_amdgcn_readfirstlane((int)(mask >> 32));
        unsigned long long steps = lo | (unsigned long long)hi << 32;
        if (!steps) continue;
        const size_t b = (size_t)p.w;
        const float wx = (float)(p.x * 8 + lx) * vs, wy = (float)(p.y * 8 + ly) * vs;
        const float wz[2] = {(float)(p.z * 8 + lz0) * vs, (float)(p.z * 8 + lz0 + 4) * vs};
        RefuseVoxel v[2];
        unsigned int word[2] = {0u, 0u};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const size_t vi = b * LF_BLOCK3 + (size_t)(t + 256 * h);
            v[h].changed = false;
            v[h].col[0] = v[h].col[1] = v[h].col[2] = 0.0f;
            if constexpr (kMixed) {
                word[h] = wd[vi];
                v[h].w = weight_value(word_code(word[h]));
                v[h].sdf = v[h].w > 0.0f ? half_bits_to_float(sdf16[vi]) : 0.0f;
#pragma unroll
                for (int k = 0; k < 3; ++k) v[h].col[k] = (float)word_channel(word[h], k);
            } else {
                v[h].w = m.weight[vi];
                v[h].sdf = v[h].w > 0.0f ? unpack_sdf(m.sdf[vi]) : 0.0f;
                if (kColour) {
                    const unsigned char *c = m.rgb + b * (3 * LF_BLOCK3) + (size_t)(t + 256 * h);
                    v[h].col[0] = c[0]; v[h].col[1] = c[LF_BLOCK3]; v[h].col[2] = c[2 * LF_BLOCK3];
                }
            }
        }
        RefuseProj pr[2];
        float4 smp[2];
        // step j's projections and sample loads
        auto look = [&](int j) {
            float T[12];
#pragma unroll
            for (int c = 0; c < 12; ++c) T[c] = s_pose[j][c];
            const float4 *samples = a.samples[j < a.n ? j : j - a.n];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                pr[h] = refuse_project<kMixed>(a, T, wx, wy, wz[h]);
                smp[h] = at_byte(samples, vgpr_offset(16u * pr[h].pix));
            }
        };
        bool use[2];
        float sd[2], wt[2];
        unsigned int rgb[2];
        // the update's selection: in the image, depth within the range, sdf >= -truncation
        auto arrive = [&]() {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float d = smp[h].x;
                sd[h] = d - pr[h].z;
                // a NaN depth and an infinite z fail the last
                use[h] = !(d > zmax) & !(d < zmin) & (sd[h] >= -m.truncation);
                wt[h] = smp[h].y;
                rgb[h] = __float_as_uint(smp[h].z);
            }
        };
        auto apply = [&](bool put_in) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
                if (use[h])
                    refuse_step<kColour, kMixed>(v[h], fminf(1.0f, sd[h] * m.inv_truncation), wt[h], rgb[h], put_in);
        };
        int j = __builtin_ctzll(steps);
        look(j);
        arrive();
        while ((steps &= steps - 1ull) != 0ull) {
            const int next = __builtin_ctzll(steps);
            look(next);
            apply(j >= a.n);
            j = next;
            arrive();
        }
        apply(j >= a.n);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (!v[h].changed) continue;
            const unsigned int o = (unsigned int)(t + 256 * h);
            const size_t vi = b * LF_BLOCK3 + o;
            const float w = v[h].w, sdf = v[h].sdf;
            if constexpr (kMixed) {
                unsigned int colour = word[h] & ~0xFFu;
                if (kColour)
                    colour = word_colour_bits((unsigned int)(int)v[h].col[0], (unsigned int)(int)v[h].col[1],
                                              (unsigned int)(int)v[h].col[2]);
                // a voxel left with a positive weight stays seen (the smallest
                // code stands for weights below it); none left: unseen
                const unsigned int code =
                    w > 0.0f ? max(1u, weight_code_sr(fminf(w, 255.0f), voxel_rand(p.x, p.y, p.z, o, pass))) : 0u;
                sdf16[vi] = code ? float_to_half_bits(sdf) : kHalfUnseen;
                wd[vi] = code | (code ? colour : (kColour ? 0u : colour));
            } else {
                m.sdf[vi] = w > 0.0f ? pack_sdf(sdf) : kSdfUnseen;
                m.weight[vi] = w;
                if (kColour) {
                    unsigned char *c = m.rgb + b * (3 * LF_BLOCK3) + o;
                    c[0] = (unsigned char)(int)v[h].col[0];
                    c[LF_BLOCK3] = (unsigned char)(int)v[h].col[1];
                    c[2 * LF_BLOCK3] = (unsigned char)(int)v[h].col[2];
                }
            }
        }
    }
}

// one map at 640x480 / 5 mm (~40k visible blocks): 4096 workgroups measured
// 70 us, 8192 and 16384 both 66 us
int integrate_grid() { return 8192; }

int check_update_args(const lf_map_params *p, const lf_map_storage *s, const float *depth, int cols, int rows,
                      const float *pose24, const lf_intrinsics *K) {
    if (!p || !s || !depth || !pose24 || !K) return lf_set_error(LF_ERR_ARG, "null argument to update");
    if (cols <= 0 || rows <= 0) return lf_set_error(LF_ERR_ARG, "bad image size %dx%d", cols, rows);
    return LF_OK;
}

}  // namespace

int lf_update_ev(const lf_map_params *p, const lf_map_storage *s, const float *depth, const float *nmap,
                 const unsigned char *rgb, int cols, int rows, const float *pose24, const lf_intrinsics *K,
                 hipStream_t st, bool weighted, hipEvent_t e0, hipEvent_t e1, const float *samples) {
    if (int rc = lf_check_storage(s, p)) return rc;
    const MapDev m = make_dev(p, s);
    dim3 g((cols + 15) / 16, (rows + 15) / 16);
    const bool mixed = p->precision == LF_PRECISION_MIXED;
    if (mixed) k_alloc<true, true><<<g, 256, 0, st>>>(m, depth, cols, rows, pose24, *K);
    else k_alloc<true, false><<<g, 256, 0, st>>>(m, depth, cols, rows, pose24, *K);
    LF_LAUNCH_CHECK();
    if (mixed) k_visible<false, true><<<visible_grid(p), kVisThreads, 0, st>>>(m, pose24, *K, cols, rows);
    else k_visible<false, false><<<visible_grid(p), kVisThreads, 0, st>>>(m, pose24, *K, cols, rows);
    LF_LAUNCH_CHECK();
    const int G = integrate_grid();
    if (e0) LF_HIP_CHECK(hipEventRecord(e0, st));
    const float4 *smp = reinterpret_cast<const float4 *>(samples);
    if (p->precision == LF_PRECISION_MIXED) {
        // the frame's packed samples (DeviceImage) or separate depth / normal / colour
        if (weighted && smp) {
            if (rgb) k_integrate<true, true, true, true><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K, smp);
            else k_integrate<true, false, true, true><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K, smp);
        } else if (weighted) {
            if (rgb) k_integrate<true, true, false, true><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K);
            else k_integrate<true, false, false, true><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K);
        } else {
            if (rgb) k_integrate<false, true, false, true><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K);
            else k_integrate<false, false, false, true><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K);
        }
    } else if (weighted && smp) {
        if (rgb) k_integrate<true, true, true><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K, smp);
        else k_integrate<true, false, true><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K, smp);
    } else if (weighted) {
        if (rgb) k_integrate<true, true><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K);
        else k_integrate<true, false><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K);
    } else {
        if (rgb) k_integrate<false, true><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K);
        else k_integrate<false, false><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K);
    }
    LF_LAUNCH_CHECK();
    if (e1) LF_HIP_CHECK(hipEventRecord(e1, st));
    return LF_OK;
}

int lf_deintegrate_ev(const lf_map_params *p, const lf_map_storage *s, const float *depth, const float *nmap,
                      const unsigned char *rgb, int cols, int rows, const float *pose24, const lf_intrinsics *K,
                      hipStream_t st, const float *samples) {
    if (int rc = lf_check_storage(s, p)) return rc;
    const MapDev m = make_dev(p, s);
    dim3 g((cols + 15) / 16, (rows + 15) / 16);
    const bool mixed = p->precision == LF_PRECISION_MIXED;
    if (mixed) k_alloc<false, true><<<g, 256, 0, st>>>(m, depth, cols, rows, pose24, *K);
    else k_alloc<false, false><<<g, 256, 0, st>>>(m, depth, cols, rows, pose24, *K);
    LF_LAUNCH_CHECK();
    if (mixed) k_visible<false, true><<<visible_grid(p), kVisThreads, 0, st>>>(m, pose24, *K, cols, rows);
    else k_visible<false, false><<<visible_grid(p), kVisThreads, 0, st>>>(m, pose24, *K, cols, rows);
    LF_LAUNCH_CHECK();
    const int G = integrate_grid();
    const float4 *smp = reinterpret_cast<const float4 *>(samples);
    if (p->precision == LF_PRECISION_MIXED) {
        if (smp) {
            if (rgb) k_deintegrate<true, true, true><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K, smp);
            else k_deintegrate<false, true, true><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K, smp);
        } else {
            if (rgb) k_deintegrate<true, false, true><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K, smp);
            else k_deintegrate<false, false, true><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K, smp);
        }
    } else if (smp) {
        if (rgb) k_deintegrate<true, true><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K, smp);
        else k_deintegrate<false, true><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K, smp);
    } else {
        if (rgb) k_deintegrate<true, false><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K, smp);
        else k_deintegrate<false, false><<<G, 256, 0, st>>>(m, depth, nmap, rgb, cols, rows, pose24, *K, smp);
    }
    LF_LAUNCH_CHECK();
    return LF_OK;
}

size_t lf_fuse_job_bytes(void) { return sizeof(FuseJob); }

int lf_update_batch_make(const LfFuseItem *items, int n, void *jobs_host, LfFuseBatchDims *dims) {
    if (!items || n <= 0 || n > 65535 || !jobs_host || !dims) return lf_set_error(LF_ERR_ARG, "bad update batch");
    FuseJob *J = static_cast<FuseJob *>(jobs_host);
    LfFuseBatchDims d = {};
    d.n = n;
    for (int i = 0; i < n; ++i) {
        const LfFuseItem &it = items[i];
        FuseJob &j = J[i];
        j = FuseJob{};
        if (!it.enabled) continue;  // tiles 0: every kernel skips this map
        if (!it.p || !it.s || !it.depth || !it.samples || !it.pose24 || !it.K || it.cols <= 0 || it.rows <= 0)
            return lf_set_error(LF_ERR_ARG, "bad update batch item %d", i);
        if (int rc = lf_check_storage(it.s, it.p)) return rc;
        const int mixed = it.p->precision == LF_PRECISION_MIXED;
        if (d.any && mixed != d.mixed)
            return lf_set_error(LF_ERR_ARG, "update batch item %d: maps of one batch share one precision", i);
        d.any = 1;
        d.mixed = mixed;
        j.m = make_dev(it.p, it.s);
        j.depth = it.depth;
        j.samples = reinterpret_cast<const float4 *>(it.samples);
        j.rgb = it.rgb;
        j.pose24 = it.pose24;
        j.K = *it.K;
        j.cols = it.cols;
        j.rows = it.rows;
        j.tiles_x = (it.cols + 15) / 16;
        j.tiles_y = (it.rows + 15) / 16;
        j.vis_grid = visible_grid(it.p);
        d.tiles_max = std::max(d.tiles_max, j.tiles_x * j.tiles_y);
        d.vis_grid_max = std::max(d.vis_grid_max, j.vis_grid);
    }
    // the single launch's 8192 workgroups shared out, at least 2048 per map
    // (16 mixed maps, frames 10-49, 5 alternating runs: 1024 / 2048 / 4096
    // per map gave 7376 / 7433 / 7429 frames/s aggregate)
    d.integrate_grid = std::max(2048, integrate_grid() / n);
    *dims = d;
    return LF_OK;
}

int lf_update_batch_launch(const void *jobs_dev, const LfFuseBatchDims &d, hipStream_t st, hipEvent_t e0,
                           hipEvent_t e1) {
    if (!jobs_dev || d.n <= 0) return lf_set_error(LF_ERR_ARG, "bad update batch launch");
    if (!d.any) return LF_OK;
    const FuseJob *J = static_cast<const FuseJob *>(jobs_dev);
    if (d.mixed) {
        k_alloc_batch<true><<<dim3(d.tiles_max, d.n), 256, 0, st>>>(J);
        LF_LAUNCH_CHECK();
        k_visible_batch<true><<<dim3(d.vis_grid_max, d.n), kVisThreads, 0, st>>>(J);
    } else {
        k_alloc_batch<false><<<dim3(d.tiles_max, d.n), 256, 0, st>>>(J);
        LF_LAUNCH_CHECK();
        k_visible_batch<false><<<dim3(d.vis_grid_max, d.n), kVisThreads, 0, st>>>(J);
    }
    LF_LAUNCH_CHECK();
    if (e0) LF_HIP_CHECK(hipEventRecord(e0, st));
    if (d.mixed) k_integrate_batch<true><<<dim3(d.integrate_grid, d.n), 256, 0, st>>>(J);
    else k_integrate_batch<false><<<dim3(d.integrate_grid, d.n), 256, 0, st>>>(J);
    LF_LAUNCH_CHECK();
    if (e1) LF_HIP_CHECK(hipEventRecord(e1, st));
    return LF_OK;
}

// The three launches of a re-fusion (the mask array cleared before them).
static int refuse_launch(const lf_map_params *p, const RefuseArgs &a, int colour, hipStream_t st) {
    LF_LAUNCH_CHECK();  // the mask clear
    const bool mixed = p->precision == LF_PRECISION_MIXED;
    const dim3 g(((a.cols + 15) / 16) * ((a.rows + 15) / 16), 2 * a.n);
    if (mixed) k_refuse_alloc<true><<<g, 256, 0, st>>>(a);
    else k_refuse_alloc<false><<<g, 256, 0, st>>>(a);
    LF_LAUNCH_CHECK();
    const int V = std::min(8 * kVisGrid, std::max(1, (p->num_blocks + kRefuseVisThreads / 4 - 1) / (kRefuseVisThreads / 4)));
    if (mixed) k_refuse_visible<true><<<V, kRefuseVisThreads, 0, st>>>(a);
    else k_refuse_visible<false><<<V, kRefuseVisThreads, 0, st>>>(a);
    LF_LAUNCH_CHECK();
    const int G = integrate_grid();
    if (mixed) {
        if (colour) k_refuse<true, true><<<G, 256, 0, st>>>(a);
        else k_refuse<false, true><<<G, 256, 0, st>>>(a);
    } else {
        if (colour) k_refuse<true, false><<<G, 256, 0, st>>>(a);
        else k_refuse<false, false><<<G, 256, 0, st>>>(a);
    }
    LF_LAUNCH_CHECK();
    return LF_OK;
}

int lf_refuse_ev(const lf_map_params *p, const lf_map_storage *s, const float *const *depth,
                 const float *const *samples, const float *const *old_pose24, const float *const *new_pose24, int n,
                 int cols, int rows, const lf_intrinsics *K, int colour, hipStream_t st) {
    if (!p || !s || !depth || !samples || !old_pose24 || !new_pose24 || !K)
        return lf_set_error(LF_ERR_ARG, "null argument to keyframe re-fusion");
    if (n < 1 || n > kMaxRefuse)
        return lf_set_error(LF_ERR_ARG, "keyframe re-fusion takes 1..%d keyframes, not %d", kMaxRefuse, n);
    if (cols <= 0 || rows <= 0) return lf_set_error(LF_ERR_ARG, "bad image size %dx%d", cols, rows);
    if (int rc = lf_check_storage(s, p)) return rc;
    if (colour && p->precision != LF_PRECISION_MIXED && !s->rgb)
        return lf_set_error(LF_ERR_ARG, "colour re-fusion needs the map's colour planes");
    RefuseArgs a = {};
    a.m = make_dev(p, s);
    for (int k = 0; k < n; ++k) {
        if (!depth[k] || !samples[k] || !old_pose24[k] || !new_pose24[k])
            return lf_set_error(LF_ERR_ARG, "null input of keyframe %d", k);
        a.depth[k] = depth[k];
        a.samples[k] = reinterpret_cast<const float4 *>(samples[k]);
        a.old24[k] = old_pose24[k];
        a.new24[k] = new_pose24[k];
    }
    a.n = n;
    a.cols = cols;
    a.rows = rows;
    a.K = *K;
    // the masks per slot and per listed block, the tiles' depths: stream-ordered device memory for the call's length
    const size_t E = (size_t)p->num_entries, B = (size_t)p->num_blocks;
    void *mask = nullptr;
    const size_t F2 = ((size_t)n * far_tiles(cols) * far_tiles(rows) + 1) / 2;  // two to a word
    LF_HIP_CHECK(hipMallocAsync(&mask, (E + F2 + B) * sizeof(unsigned long long), st));
    a.slot_mask = static_cast<unsigned long long *>(mask);
    a.list_mask = a.slot_mask + E + F2;
    a.tile_far = reinterpret_cast<int *>(a.slot_mask + E);
    k_fill_u64<<<(int)std::min<size_t>(4096, (E + F2 + 255) / 256), 256, 0, st>>>(a.slot_mask, E + F2);
    const int rc = refuse_launch(p, a, colour, st);
    const hipError_t ef = hipFreeAsync(mask, st);
    if (rc) return rc;
    if (ef != hipSuccess) return lf_set_error(LF_ERR_HIP, "hipFreeAsync failed: %s", hipGetErrorString(ef));
    return LF_OK;
}

extern "C" int lf_deintegrate_weighted(const lf_map_params *p, const lf_map_storage *s, const float *depth,
                                       const float *nmap, const unsigned char *rgb, int cols, int rows,
                                       const float *pose24, const lf_intrinsics *K, void *stream) {
    int rc = check_update_args(p, s, depth, cols, rows, pose24, K);
    if (rc) return rc;
    if (!nmap) return lf_set_error(LF_ERR_ARG, "deintegrate_weighted needs a normal map");
    return lf_deintegrate_ev(p, s, depth, nmap, rgb, cols, rows, pose24, K, lf_stream(stream), nullptr);
}

__global__ void k_reset_visible(MapDev m) {
    if (threadIdx.x == 0 && blockIdx.x == 0) m.counters[LF_CNT_VISIBLE] = 0u;
}

int lf_select_visible_ev(const lf_map_params *p, const lf_map_storage *s, const float *pose24, const lf_intrinsics *K,
                         int cols, int rows, hipStream_t st) {
    if (int rc = lf_check_storage(s, p)) return rc;
    const MapDev m = make_dev(p, s);
    k_reset_visible<<<1, 64, 0, st>>>(m);
    LF_LAUNCH_CHECK();
    if (p->precision == LF_PRECISION_MIXED)
        k_visible<true, true><<<visible_grid(p), kVisThreads, 0, st>>>(m, pose24, *K, cols, rows);
    else
        k_visible<true, false><<<visible_grid(p), kVisThreads, 0, st>>>(m, pose24, *K, cols, rows);
    LF_LAUNCH_CHECK();
    return LF_OK;
}

extern "C" int lf_select_visible(const lf_map_params *p, const lf_map_storage *s, const float *pose24,
                                 const lf_intrinsics *K, int cols, int rows, unsigned int *count_out, void *stream) {
    if (!p || !s || !pose24 || !K || cols <= 0 || rows <= 0)
        return lf_set_error(LF_ERR_ARG, "bad arguments to lf_select_visible");
    hipStream_t st = lf_stream(stream);
    if (int rc = lf_select_visible_ev(p, s, pose24, K, cols, rows, st)) return rc;
    if (count_out) {
        LF_HIP_CHECK(hipMemcpyAsync(count_out, s->counters + LF_CNT_VISIBLE, sizeof(unsigned int),
                                    hipMemcpyDeviceToHost, st));
        LF_HIP_CHECK(hipStreamSynchronize(st));
    }
    return LF_OK;
}

extern "C" int lf_update_weighted(const lf_map_params *p, const lf_map_storage *s, const float *depth,
                                  const float *nmap, const unsigned char *rgb, int cols, int rows,
                                  const float *pose24, const lf_intrinsics *K, void *stream) {
    int rc = check_update_args(p, s, depth, cols, rows, pose24, K);
    if (rc) return rc;
    if (!nmap) return lf_set_error(LF_ERR_ARG, "update_weighted needs a normal map");
    return lf_update_ev(p, s, depth, nmap, rgb, cols, rows, pose24, K, lf_stream(stream), true, nullptr, nullptr);
}

extern "C" int lf_update(const lf_map_params *p, const lf_map_storage *s, const float *depth,
                         const unsigned char *rgb, int cols, int rows, const float *pose24, const lf_intrinsics *K,
                         void *stream) {
    int rc = check_update_args(p, s, depth, cols, rows, pose24, K);
    if (rc) return rc;
    return lf_update_ev(p, s, depth, nullptr, rgb, cols, rows, pose24, K, lf_stream(stream), false, nullptr,
                        nullptr);
}
