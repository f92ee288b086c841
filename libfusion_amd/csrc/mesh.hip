// Marching-cubes mesh extraction over every allocated voxel block.
//
// Reference: src/voxel_hashing/scene_mesh.cu — BuildVertexArray (:14-248:
// read_sdf_list :70-106, interpolate_sdf :108-117, make_vertex :119-209,
// emitter :211-247), BuildVertexAndColourArray (:353-588), hosts
// create_mesh_vertex_only / _with_normal / _with_colour (:260-351,600-643);
// tables include/voxel_hashing/device_tables.h.
//
// MI355X design: one wavefront per block, eight blocks per workgroup.
//  * The block's 9x9x9 corner lattice (its own 512 voxels plus the faces of the
//    7 +x/+y/+z neighbours) is staged in LDS as 2-byte sdf codes: five loads a
//    lane (the own block is one 16-byte load).  Without colours the code alone
//    decides validity (weight 0 <=> the unseen code), so the 4-byte weights are
//    not read.
//  * Each lane classifies the 8 cubes of one (x, y) column, sharing the corner
//    layers between them; the counts give every cube's place with ballots.
//  * The triangles are emitted one lane each, not one cube each: cubes append
//    (cube, triangle) entries to a list in LDS and 64 at a time become
//    vertices.  (A lane per cube looped over up to 5 triangles, its 12 edge
//    vertices in scratch memory for want of constant indices.)
//  * One atomic reserves the output of the workgroup's eight blocks: the
//    appends to one counter serialise.
//  Measured on 18k blocks / 2.43 M triangles with normals (8 mm, mixed, 175 MB
//  out): 406 -> 95 us.  Whole calls, the count read: vertices 238 -> 96 us (FP32 88),
//  normals 365 -> 109 (FP32 364 -> 105), colours, each vertex's gathered where it is
//  emitted, 320 -> 109 (FP32 354 -> 108).  Half of the kernel is the chain block ->
//  neighbours -> lattice -> reservation (49 us with the emission left out), so it is
//  held to 64 VGPRs for 8 wavefronts per SIMD; stores through LDS, contiguous
//  over the wavefront, cost that occupancy and took 114 us, and the eight
//  wavefronts sharing one triangle list 138 us.
#include "lf_common.h"
#include "mc_tables.h"

using namespace lf;

namespace {

// The triangle table by triangle: entry ci * 5 + k holds the three edges of
// triangle k of cube case ci, each as the two corners it joins (first, second
// in the direction interpolate_sdf walks it), a corner as bits x | y << 1 |
// z << 2; 6 bits an edge.  ntri[ci]: the case's triangles.
struct TriTable {
    unsigned int edges[256 * 5];
    unsigned char ntri[256];
};
constexpr TriTable make_tri_table() {
    constexpr signed char tri[256][16] = LF_MC_TRI_TABLE_DATA;
    // corner k of the cube (scene_mesh.cu:119-209) and the corners of its 12 edges
    constexpr unsigned int corner[8] = {0, 1, 3, 2, 4, 5, 7, 6};
    constexpr int first[12] = {0, 1, 2, 3, 4, 5, 6, 7, 0, 1, 2, 3}, second[12] = {1, 2, 3, 0, 5, 6, 7, 4, 4, 5, 6, 7};
    TriTable t = {};
    for (int ci = 0; ci < 256; ++ci) {
        int n = 0;
        while (n < 5 && tri[ci][3 * n] != -1) {
            unsigned int d = 0;
            for (int k = 0; k < 3; ++k) {
                const int e = tri[ci][3 * n + k];
                d |= (corner[first[e]] | corner[second[e]] << 3) << (6 * k);
            }
            t.edges[ci * 5 + n] = d;
            ++n;
        }
        t.ntri[ci] = (unsigned char)n;
    }
    return t;
}
__constant__ TriTable c_tri = make_tri_table();

struct MeshDev {
    const unsigned long long *keys;
    const int *slot_block;
    const int *block_pos;
    const int *block_dir;
    const short *sdf;
    const float *weight;
    const unsigned char *rgb;
    unsigned int *counters;
    int num_buckets, num_entries, num_blocks;
    float voxel_size;
};

__global__ void k_mesh_begin(unsigned int *counters) { counters[LF_CNT_TRIANGLES] = 0u; }

LF_DEV float interp_edge(float v1, float v2) {  // interpolate_sdf (scene_mesh.cu:108-117)
    // (double)x < 1e-6 for a float x is x <= 1e-6f, the largest float below 1e-6
    if (fabsf(0.0f - v1) <= 1e-6f) return 0.0f;
    if (fabsf(0.0f - v2) <= 1e-6f) return 1.0f;
    if (fabsf(v1 - v2) <= 1e-6f) return 0.0f;
    return (0.0f - v1) / (v2 - v1);
}

constexpr int kMeshWaves = 8;     // wavefronts (blocks) of a workgroup
constexpr int kMeshGrid = 1024;   // workgroups resident at once: 64 VGPRs and 30 KB of LDS, four to a CU
constexpr int kLattice = 9 * 9 * 9;
constexpr int kMaxLayer = 64 * 5;  // triangles of one 8x8 layer of cubes
constexpr int kList = 64 + kMaxLayer;

struct MeshWave {  // one wavefront's LDS
    unsigned short sdf[kLattice + 7];
    int nb[8];                // pool blocks of the 2x2x2 neighbourhood, -1: none
    unsigned int list[kList];  // cube | triangle << 9 | case << 12
};

// LDS written by other lanes of this wavefront: its LDS operations run in
// order, so only the compiler has to keep them so.
LF_DEV void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

LF_DEV unsigned int lanes_below(unsigned long long mask) {
    return __builtin_amdgcn_mbcnt_hi((unsigned int)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned int)mask, 0u));
}

// A voxel's sdf code, or the unseen code where the mesh takes it for invalid:
// weight 0, with colours (kMode 2) a weight of at most 1e-3.
template <int kMode, bool kMixed>
LF_DEV unsigned short corner_code(const MeshDev &m, size_t vi) {
    constexpr unsigned short unseen = kMixed ? kHalfUnseen : (unsigned short)kSdfUnseen;
    const unsigned short c = reinterpret_cast<const unsigned short *>(m.sdf)[vi];
    if constexpr (kMode == 2) {
        const float w =
            kMixed ? weight_value(word_code(reinterpret_cast<const unsigned int *>(m.weight)[vi])) : m.weight[vi];
        return (double)w > 1e-3 ? c : unseen;
    }
    return c;
}

// Block blk_i at P into the wavefront's lattice.
template <int kMode, bool kMixed>
LF_DEV void stage_block(const MeshDev &m, MeshWave &s, int blk_i, int4 P, int lane) {
    constexpr unsigned short unseen = kMixed ? kHalfUnseen : (unsigned short)kSdfUnseen;
    const unsigned short *sdf16 = reinterpret_cast<const unsigned short *>(m.sdf);
    // own rows: lane l holds the 8 voxels of row (y, z) = (l & 7, l >> 3)
    const size_t own = (size_t)blk_i * LF_BLOCK3 + 8 * lane;
    unsigned short row[8];
    {
        unsigned int q[4];  // one 16-byte load; a caller's plane need only be aligned to its codes
        __builtin_memcpy(q, sdf16 + own, 16);
#pragma unroll
        for (int k = 0; k < 8; ++k) row[k] = (unsigned short)(q[k >> 1] >> (16 * (k & 1)));
        if constexpr (kMode == 2) {
#pragma unroll
            for (int k = 0; k < 8; ++k) row[k] = corner_code<kMode, kMixed>(m, own + k);
        }
    }
    int nb = blk_i;
    if (lane > 0 && lane < 8) {
        const int x = P.x + (lane & 1), y = P.y + ((lane >> 1) & 1), z = P.z + (lane >> 2);
        const int cell = dir_cell(x, y, z);
        nb = cell >= 0 ? m.block_dir[cell] : find_block(m.keys, m.slot_block, x, y, z, m.num_buckets, m.num_entries);
    }
    if (lane < 8) s.nb[lane] = nb;
    const int a = lane & 7, b = lane >> 3;
    {
        unsigned short *o = s.sdf + 9 * a + 81 * b;
#pragma unroll
        for (int k = 0; k < 8; ++k) o[k] = row[k];
    }
    // the three faces (64 corners each), then the three edges and the corner
    const int nx = __shfl(nb, 1), ny = __shfl(nb, 2), nz = __shfl(nb, 4);
    const auto at = [&](int n, int l) {
        return n < 0 ? unseen : corner_code<kMode, kMixed>(m, (size_t)n * LF_BLOCK3 + l);
    };
    s.sdf[8 + 9 * a + 81 * b] = at(nx, b << 6 | a << 3);
    s.sdf[a + 72 + 81 * b] = at(ny, b << 6 | a);
    s.sdf[a + 9 * b + 648] = at(nz, b << 3 | a);
    if (lane < 25) {
        const int e = lane < 24 ? (b == 0 ? 3 : b == 1 ? 5 : 6) : 7;  // the neighbour across two (three) faces
        const int ex = e & 1 ? 8 : a, ey = e & 2 ? 8 : a, ez = e & 4 ? 8 : a;
        s.sdf[ex + 9 * ey + 81 * ez] = at(__shfl(nb, e), lidx(ex, ey, ez));
    }
}

template <bool kMixed>
LF_DEV float code_value(unsigned short c) {
    if constexpr (kMixed) return half_bits_to_float(c);
    else return unpack_sdf((short)c);
}

// mode 0: vertices, 1: + flat normals, 2: + corner colours.  kMixed: FP16
// sdf and 8-bit weight codes.
template <int kMode, bool kMixed>
__global__ __launch_bounds__(64 * kMeshWaves, 8) void k_mesh(MeshDev m, float *__restrict__ vtx,
                                                             float *__restrict__ nrm, unsigned char *__restrict__ col,
                                                             unsigned int max_tri) {
    constexpr unsigned short unseen = kMixed ? kHalfUnseen : (unsigned short)kSdfUnseen;
    __shared__ TriTable s_tri;
    __shared__ MeshWave s_wave[kMeshWaves];
    __shared__ unsigned int s_cnt[2][kMeshWaves], s_base[2];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    MeshWave &s = s_wave[wave];
    {
        const unsigned int *src = reinterpret_cast<const unsigned int *>(&c_tri);
        unsigned int *dst = reinterpret_cast<unsigned int *>(&s_tri);
        for (int i = tid; i < (int)(sizeof(TriTable) / 4); i += 64 * kMeshWaves) dst[i] = src[i];
    }
    const unsigned int nblk = min(m.counters[LF_CNT_ALLOCATED], (unsigned int)m.num_blocks);
    const float vs = m.voxel_size;
    __syncthreads();
    int par = 0;  // the counts of one round are read while the next round's are written
    for (unsigned int b0 = blockIdx.x * kMeshWaves; b0 < nblk; b0 += gridDim.x * kMeshWaves, par ^= 1) {
        const unsigned int blk_i = b0 + wave;
        int4 P = make_int4(0, 0, 0, 0);
        unsigned int cases[2] = {0u, 0u};  // the lane's 8 cube cases, one byte each; 0: no triangles
        unsigned int total = 0;
        if (blk_i < nblk) {
            P = reinterpret_cast<const int4 *>(m.block_pos)[blk_i];
            stage_block<kMode, kMixed>(m, s, (int)blk_i, P, lane);
            wave_lds_fence();
            // the column of cubes at (x, y): corner layer z is the top of cube
            // z - 1 and the bottom of cube z
            const unsigned short *c = s.sdf + (lane & 7) + 9 * (lane >> 3);
            unsigned int below = 0;
            bool below_ok = false;
#pragma unroll
            for (int z = 0; z < 9; ++z) {
                const unsigned short q[4] = {c[81 * z], c[81 * z + 1], c[81 * z + 10], c[81 * z + 9]};
                unsigned int bits = 0;
                bool ok = true;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    ok = ok && q[k] != unseen;
                    bits |= (code_value<kMixed>(q[k]) < 0.0f ? 1u : 0u) << k;
                }
                if (z > 0) {
                    const unsigned int ci = ok && below_ok ? below | bits << 4 : 0u;
                    cases[(z - 1) >> 2] |= ci << (8 * ((z - 1) & 3));
                    const unsigned int n = s_tri.ntri[ci];
                    total += __popcll(__ballot(n & 1)) + 2 * __popcll(__ballot(n & 2)) + 4 * __popcll(__ballot(n & 4));
                }
                below = bits;
                below_ok = ok;
            }
        }
        if (lane == 0) s_cnt[par][wave] = total;
        __syncthreads();
        if (tid == 0) {
            unsigned int sum = 0;
#pragma unroll
            for (int w = 0; w < kMeshWaves; ++w) {
                const unsigned int c = s_cnt[par][w];
                s_cnt[par][w] = sum;
                sum += c;
            }
            s_base[par] = sum ? atomicAdd(&m.counters[LF_CNT_TRIANGLES], sum) : 0u;
        }
        __syncthreads();
        if (total == 0) continue;  // the whole wavefront
        unsigned int id = s_base[par] + s_cnt[par][wave];  // the list's first triangle
        const int bx = P.x * 8, by = P.y * 8, bz = P.z * 8;
        unsigned int len = 0;
        // cnt <= 64 triangles of the list, one lane each
        auto emit = [&](unsigned int from, unsigned int cnt) {
            const unsigned int ent = s.list[from + min((unsigned int)lane, cnt - 1)];
            const unsigned int d = s_tri.edges[(ent >> 12) * 5 + ((ent >> 9) & 7)];
            const int lx = ent & 7, ly = (ent >> 3) & 7, lz = (ent >> 6) & 7;
            const int li = lx + 9 * ly + 81 * lz;
            const float p[3] = {(float)(bx + lx), (float)(by + ly), (float)(bz + lz)};
            f3 t3[3];
            unsigned char colour[9];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const unsigned int A = (d >> (6 * k)) & 7u, B = (d >> (6 * k + 3)) & 7u, axis = A ^ B;
                const unsigned int ax = A & 1u, ay = (A >> 1) & 1u, az = A >> 2;
                const float v1 = code_value<kMixed>(s.sdf[li + (int)(ax + 9 * ay + 81 * az)]);
                const unsigned int bx1 = B & 1u, by1 = (B >> 1) & 1u, bz1 = B >> 2;
                const float v2 = code_value<kMixed>(s.sdf[li + (int)(bx1 + 9 * by1 + 81 * bz1)]);
                float t = interp_edge(v1, v2);
                if (A & axis) t = 1.0f - t;  // an edge walked from its far end
                t3[k] = mul(f3{p[0] + (axis == 1u ? t : (float)ax), p[1] + (axis == 2u ? t : (float)ay),
                               p[2] + (axis == 4u ? t : (float)az)}, vs);
                if constexpr (kMode == 2) {  // colour of the edge's first corner
                    const int cx = lx + (int)ax, cy = ly + (int)ay, cz = lz + (int)az;
                    const size_t nb = (size_t)s.nb[(cx >> 3) | (cy >> 3) << 1 | (cz >> 3) << 2];
                    const int l = lidx(cx, cy, cz);
                    if (kMixed) {
                        const unsigned int word = reinterpret_cast<const unsigned int *>(m.weight)[nb * LF_BLOCK3 + l];
#pragma unroll
                        for (int q = 0; q < 3; ++q) colour[3 * k + q] = (unsigned char)word_channel(word, q);
                    } else {
                        const unsigned char *c = m.rgb + nb * (3 * LF_BLOCK3) + l;
                        colour[3 * k] = c[0]; colour[3 * k + 1] = c[LF_BLOCK3]; colour[3 * k + 2] = c[2 * LF_BLOCK3];
                    }
                }
            }
            // below the capacity (the count goes on beyond it)
            const bool in = (unsigned int)lane < cnt && id + lane < max_tri;
            if (vtx && in) {
                float *o = vtx + 9 * ((size_t)id + lane);
#pragma unroll
                for (int k = 0; k < 3; ++k) { o[3 * k] = t3[k].x; o[3 * k + 1] = t3[k].y; o[3 * k + 2] = t3[k].z; }
            }
            if (kMode == 1 && nrm && in) {
                const f3 n = normalised(cross(sub(t3[1], t3[0]), sub(t3[2], t3[0])));
                float *o = nrm + 9 * ((size_t)id + lane);
#pragma unroll
                for (int k = 0; k < 3; ++k) { o[3 * k] = n.x; o[3 * k + 1] = n.y; o[3 * k + 2] = n.z; }
            }
            if (kMode == 2 && col && in) {
                unsigned char *o = col + 9 * ((size_t)id + lane);
#pragma unroll
                for (int k = 0; k < 9; ++k) o[k] = colour[k];
            }
            id += cnt;
        };
        // layers of cubes appended to the list, full wavefronts of triangles
        // taken from its front as they come together (the list holds what is
        // left of one and a whole layer)
#pragma unroll 1
        for (int z = 0; z < 8; ++z) {
            const unsigned int ci = (cases[z >> 2] >> (8 * (z & 3))) & 0xFFu, n = s_tri.ntri[ci];
            const unsigned long long n1 = __ballot(n & 1), n2 = __ballot(n & 2), n4 = __ballot(n & 4);
            const unsigned int layer = __popcll(n1) + 2 * __popcll(n2) + 4 * __popcll(n4);
            if (layer == 0) continue;
            const unsigned int at = len + lanes_below(n1) + 2 * lanes_below(n2) + 4 * lanes_below(n4);
            for (unsigned int k = 0; k < n; ++k) s.list[at + k] = (unsigned int)(z << 6 | lane) | k << 9 | ci << 12;
            len += layer;
            wave_lds_fence();
            unsigned int from = 0;
            for (; len - from >= 64; from += 64) emit(from, 64);
            if (from) {  // the rest to the front
                len -= from;
                const bool mine = (unsigned int)lane < len;
                const unsigned int e = mine ? s.list[from + lane] : 0u;
                wave_lds_fence();
                if (mine) s.list[lane] = e;
                wave_lds_fence();
            }
        }
        if (len) emit(0, len);
    }
}

}  // namespace

extern "C" int lf_create_mesh(const lf_map_params *p, const lf_map_storage *s, float *vertex_out, float *normal_out,
                              unsigned char *colour_out, int max_triangles, unsigned int *triangles_out,
                              void *stream) {
    if (!p || !s || !triangles_out) return lf_set_error(LF_ERR_ARG, "null argument to create_mesh");
    if (max_triangles < 0) return lf_set_error(LF_ERR_ARG, "negative triangle capacity");
    if (normal_out && colour_out) return lf_set_error(LF_ERR_ARG, "ask for normals or colours, not both");
    if (int rc = lf_check_storage(s, p)) return rc;
    hipStream_t st = lf_stream(stream);
    MeshDev m;
    m.keys = s->keys; m.slot_block = s->slot_block; m.block_pos = s->block_pos; m.block_dir = s->block_dir;
    m.sdf = s->sdf; m.weight = s->weight; m.rgb = s->rgb; m.counters = s->counters;
    m.num_buckets = p->num_buckets; m.num_entries = p->num_entries; m.num_blocks = p->num_blocks;
    m.voxel_size = p->voxel_size;
    k_mesh_begin<<<1, 1, 0, st>>>(s->counters);
    LF_LAUNCH_CHECK();
    const int G = std::max(1, std::min((p->num_blocks + kMeshWaves - 1) / kMeshWaves, kMeshGrid));
    const unsigned int cap = (unsigned int)max_triangles;
    if (p->precision == LF_PRECISION_MIXED) {
        if (colour_out) k_mesh<2, true><<<G, 64 * kMeshWaves, 0, st>>>(m, vertex_out, nullptr, colour_out, cap);
        else if (normal_out) k_mesh<1, true><<<G, 64 * kMeshWaves, 0, st>>>(m, vertex_out, normal_out, nullptr, cap);
        else k_mesh<0, true><<<G, 64 * kMeshWaves, 0, st>>>(m, vertex_out, nullptr, nullptr, cap);
    } else {
        if (colour_out) k_mesh<2, false><<<G, 64 * kMeshWaves, 0, st>>>(m, vertex_out, nullptr, colour_out, cap);
        else if (normal_out) k_mesh<1, false><<<G, 64 * kMeshWaves, 0, st>>>(m, vertex_out, normal_out, nullptr, cap);
        else k_mesh<0, false><<<G, 64 * kMeshWaves, 0, st>>>(m, vertex_out, nullptr, nullptr, cap);
    }
    LF_LAUNCH_CHECK();
    unsigned int cnt = 0;
    LF_HIP_CHECK(hipMemcpyAsync(&cnt, s->counters + LF_CNT_TRIANGLES, sizeof(cnt), hipMemcpyDeviceToHost, st));
    LF_HIP_CHECK(hipStreamSynchronize(st));
    *triangles_out = std::min(cnt, cap);
    if (cnt > cap) return lf_set_error(LF_ERR_CAPACITY, "mesh has %u triangles, capacity %u", cnt, cap);
    return LF_OK;
}
