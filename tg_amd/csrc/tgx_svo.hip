/*
 * tgx_svo.hip — sparse voxel octree build on gfx950.
 *
 * Build (replaces tg_svo_create, tg_sparse_voxel_octree.c:466-542, a
 * single-threaded depth-first recursion on the host):
 *   1. svo_frames_k      per cluster pointer: emptiness flag and the three
 *                        cluster transforms of the reference (world->cluster
 *                        :23-60, cluster->world :62-100 and its inverse).
 *   2. per level         (node, cluster pointer) pairs; svo_expand_k runs
 *                        tg_intersect_aabb_obb_ignore_contact for the 8
 *                        children of each pair, appends the survivors to the
 *                        next level's pairs and sets their cells in its bitmap.
 *   3. svo_nodes_k       the bitmaps of all levels, one after the other, are the
 *                        nodes in (level, Morton code) order: a scan of their
 *                        popcounts numbers them, a node's children are one byte
 *                        of the next level, contiguous in child-index order.
 *      svo_pair_*_k      the leaf level's pairs sorted by (leaf, cluster
 *                        pointer): each leaf's clusters in ascending pointer
 *                        order (the reference's list order).
 *   4. svo_leaf_k        one workgroup per 32^3 leaf: the trimmed block box of
 *      svo_leaf_mats_k   each candidate cluster is point sampled in the
 *      svo_leaf_mats_few_k reference's exact fp32 order (:242-315); solid bits
 *                        collect in LDS, then the material of the first
 *                        candidate that sampled a voxel solid.
 * Traversal and GI live in tgx_gi.hip.
 */
#include "tgx_gi_dev.h"
#include "tgx_m4.h"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <vector>

/* Per-cluster-pointer transforms (rows 0..2 of each m4). */
struct svo_frame {
    float    ws2ms[12];
    float    cs2ws[12];
    float    ws2cs[12];
    uint32_t cidx;
    uint32_t lut;         /* (lut_idx & 255) << 8 */
    uint32_t pad[2];
};
static_assert(sizeof(svo_frame) == 160, "svo_frame layout");

/* rows 0..2 of m times (x, y, z, w), tg_math.c:2428-2438 order */
__device__ static inline f3 mulv(const float* m, float x, float y, float z, float w)
{
    f3 r;
    r.x = x * m[0] + y * m[1] + z * m[2] + w * m[3];
    r.y = x * m[4] + y * m[5] + z * m[6] + w * m[7];
    r.z = x * m[8] + y * m[9] + z * m[10] + w * m[11];
    return r;
}

__device__ static inline uint32_t spread3(uint32_t v)
{
    v &= 0x3FFu;
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}
__device__ static inline uint32_t compact3(uint32_t v)
{
    v &= 0x09249249u;
    v = (v | (v >> 2)) & 0x030C30C3u;
    v = (v | (v >> 4)) & 0x0300F00Fu;
    v = (v | (v >> 8)) & 0x030000FFu;
    v = (v | (v >> 16)) & 0x000003FFu;
    return v;
}
__device__ static inline uint32_t morton3(uint32_t x, uint32_t y, uint32_t z)
{
    return spread3(x) | (spread3(y) << 1) | (spread3(z) << 2);
}

/* ------------------------------------------------------------------------ */
/* tg_intersect_aabb_obb_ignore_contact against the cluster box [0,8]^3     */
/* (tg_physics.c:226-392), corners c[8] in cluster space                    */
/* ------------------------------------------------------------------------ */

__device__ static inline f3 f3_sub(f3 a, f3 b) { f3 r = {a.x - b.x, a.y - b.y, a.z - b.z}; return r; }
__device__ static inline float f3_dot(f3 a, f3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ static inline float f3_mag(f3 a) { return sqrtf(a.x * a.x + a.y * a.y + a.z * a.z); }
__device__ static inline f3 f3_normalized(f3 a)
{
    const float m = f3_mag(a);
    f3 r = {a.x / m, a.y / m, a.z / m};
    return r;
}

__device__ static bool obb_overlaps_cluster(const f3* c)
{
    bool sep;
    sep = true; for (int i = 0; i < 8; i++) sep = sep && c[i].x <= 0.0f; if (sep) return false;
    sep = true; for (int i = 0; i < 8; i++) sep = sep && c[i].x >= 8.0f; if (sep) return false;
    sep = true; for (int i = 0; i < 8; i++) sep = sep && c[i].y <= 0.0f; if (sep) return false;
    sep = true; for (int i = 0; i < 8; i++) sep = sep && c[i].y >= 8.0f; if (sep) return false;
    sep = true; for (int i = 0; i < 8; i++) sep = sep && c[i].z <= 0.0f; if (sep) return false;
    sep = true; for (int i = 0; i < 8; i++) sep = sep && c[i].z >= 8.0f; if (sep) return false;

    const f3 nxp = f3_normalized(f3_sub(c[1], c[0]));
    const f3 nyp = f3_normalized(f3_sub(c[2], c[0]));
    const f3 nzp = f3_normalized(f3_sub(c[4], c[0]));
    f3 nrm[6];
    nrm[0] = {-nxp.x, -nxp.y, -nxp.z}; nrm[1] = nxp;
    nrm[2] = {-nyp.x, -nyp.y, -nyp.z}; nrm[3] = nyp;
    nrm[4] = {-nzp.x, -nzp.y, -nzp.z}; nrm[5] = nzp;
    const float l0 = f3_mag(c[0]);
    const float l1 = f3_mag(c[7]);
    f3 n0 = {0.0f, 0.0f, 0.0f}, n1 = {0.0f, 0.0f, 0.0f};
    if (l0 != 0.0f) { n0.x = c[0].x / l0; n0.y = c[0].y / l0; n0.z = c[0].z / l0; }
    if (l1 != 0.0f) { n1.x = c[7].x / l1; n1.y = c[7].y / l1; n1.z = c[7].z / l1; }
    float dist[6];
    dist[0] = l0 * f3_dot(n0, nrm[0]);
    dist[1] = l1 * f3_dot(n1, nrm[1]);
    dist[2] = l0 * f3_dot(n0, nrm[2]);
    dist[3] = l1 * f3_dot(n1, nrm[3]);
    dist[4] = l0 * f3_dot(n0, nrm[4]);
    dist[5] = l1 * f3_dot(n1, nrm[5]);
    for (int p = 0; p < 6; p++) {
        sep = true;
        for (int i = 0; i < 8 && sep; i++) {
            const f3 pt = {(i & 1) ? 8.0f : 0.0f, (i & 2) ? 8.0f : 0.0f, (i & 4) ? 8.0f : 0.0f};
            sep = (f3_dot(nrm[p], pt) - dist[p]) >= 0.0f;
        }
        if (sep) return false;
    }
    return true;
}

/* ------------------------------------------------------------------------ */
/* Build kernels                                                            */
/* ------------------------------------------------------------------------ */

__global__ __launch_bounds__(256) void svo_frames_k(const tgx_object* __restrict__ objects,
                                                    const uint32_t* __restrict__ cptrs,
                                                    const uint32_t* __restrict__ c2o,
                                                    const uint32_t* __restrict__ bits, uint32_t n_cptr,
                                                    svo_frame* __restrict__ frames, uint32_t* __restrict__ nonempty)
{
    const uint32_t cp = blockIdx.x * blockDim.x + threadIdx.x;
    if (cp >= n_cptr) return;
    const uint32_t cidx = cptrs[cp];
    uint32_t any = 0;
    for (int i = 0; i < 16; i++) any |= bits[(size_t)cidx * 16u + i];
    nonempty[cp] = any ? 1u : 0u;
    const tgx_object ob = objects[c2o[cidx]];
    const uint32_t rel = cp - ob.first_cluster_pointer;
    const uint32_t nx = ob.n_cluster_pointers_per_dim[0], ny = ob.n_cluster_pointers_per_dim[1];
    const uint32_t rx = rel % nx, ry = (rel / nx) % ny, rz = rel / (nx * ny);
    const tgx_m4 w2c = tgx_world_to_cluster(ob.rotation, ob.translation, ob.n_cluster_pointers_per_dim, rx, ry, rz);
    const tgx_m4 c2w = tgx_cluster_to_world(ob.rotation, ob.translation, ob.n_cluster_pointers_per_dim, rx, ry, rz);
    const tgx_m4 w2c2 = tgx_m4_inverse(c2w);
    svo_frame f;
    for (int r = 0; r < 3; r++)
        for (int c = 0; c < 4; c++) {
            f.ws2ms[4 * r + c] = TGX_M(w2c, r, c);
            f.cs2ws[4 * r + c] = TGX_M(c2w, r, c);
            f.ws2cs[4 * r + c] = TGX_M(w2c2, r, c);
        }
    f.cidx = cidx;
    f.lut = (ob.lut_idx & 0xFFu) << 8;
    f.pad[0] = f.pad[1] = 0u;
    frames[cp] = f;
}

/* Packed node coordinates: x | y << 10 | z << 20. */
__device__ static inline void unpack(uint32_t p, uint32_t& x, uint32_t& y, uint32_t& z)
{
    x = p & 0x3FFu; y = (p >> 10) & 0x3FFu; z = p >> 20;
}

/* The nodes of all levels as one bitmap: level l's 8^l cells in Morton order
 * from word node_word(l), so bits in word order are the nodes in canonical
 * order and a node's children are one byte of the next level. */
__host__ __device__ static inline uint32_t level_words(uint32_t l) { return l < 2u ? 1u : 1u << (3u * l - 5u); }
__host__ __device__ static inline uint32_t node_word(uint32_t l)
{
    uint32_t w = 0u;
    for (uint32_t k = 0; k < l; k++) w += level_words(k);
    return w;
}

/* Counters of a build (u32): pairs of level l at l, then the summary the host
 * reads: first node of level l at SVO_CNT_BASE + l, all nodes after the last;
 * leaves that an update took over at SVO_CNT_REUSED; at SVO_CNT_MANY the leaves
 * that are svo_leaf_mats_k's (leaf_few); at SVO_CNT_WRAP whether the leaves'
 * solid voxels are more than the 32-bit material offsets hold. */
#define SVO_CNT_BASE 16u
#define SVO_CNT_REUSED 31u
#define SVO_CNT_MANY 30u
#define SVO_CNT_WRAP 29u
#define SVO_CNT_N    32u

/* Children of the level's (node, cluster pointer) pairs: eight lanes per pair,
 * one child each (tg_intersect_aabb_obb_ignore_contact). The survivors are
 * appended to the next level's pairs, in no order (the leaf level's are sorted
 * once), up to cap of them; *n_out counts all. Their cells, one byte per pair,
 * are set in the level's bitmap. Level 0 takes the non-empty cluster pointers
 * themselves (coord null).
 * What bounds it is the bitmap's atomics, which leave the XCD: at depth 11
 * and 60 k leaf pairs the last level takes 77 us with an atomic per child, 60
 * with one per pair, and 25 where each block gathers them in LDS and adds the
 * words that are not yet set. That is done up to 8192 words (level 6); beyond,
 * a block would clear and read more words than it has pairs. Two blocks of 16
 * waves per CU loop over the pairs, so that there are few maps to add (on 18 M
 * clusters a level takes 2.6 ms, where a lane per pair took 0.7 for the tests
 * alone). All levels: 116 us, and no host round trip, for what took 145 us in the
 * tests alone (a lane per pair, its eight children in turn) and 295 us in scans
 * and sorts. */
#define EXPAND_BLOCK 1024u
#define EXPAND_PAIRS (EXPAND_BLOCK / 8u)
#define EXPAND_LDS_WORDS 8192u
#define EXPAND_BLOCKS 512u
__global__ __launch_bounds__(EXPAND_BLOCK) void svo_expand_k(const uint32_t* __restrict__ coord,
                                                             const uint32_t* __restrict__ cptr,
                                                             const uint32_t* __restrict__ nonempty,
                                                             const uint32_t* __restrict__ n_in, uint32_t n_max,
                                                             const svo_frame* __restrict__ frames, float mnx, float mny,
                                                             float mnz, float side, uint32_t* __restrict__ n_out,
                                                             uint32_t* __restrict__ out_coord,
                                                             uint32_t* __restrict__ out_cptr, uint32_t cap,
                                                             uint32_t* __restrict__ map, uint32_t map_words)
{
    __shared__ uint32_t s_map[EXPAND_LDS_WORDS];
    const bool lds = map_words <= EXPAND_LDS_WORDS;
    const uint32_t n_all = coord ? *n_in : n_max, n = n_all < n_max ? n_all : n_max;
    if (blockIdx.x * EXPAND_PAIRS >= n) return;
    if (lds) {
        for (uint32_t w = threadIdx.x; w < map_words; w += EXPAND_BLOCK) s_map[w] = 0u;
        __syncthreads();
    }
    const uint32_t c = threadIdx.x & 7u;
    for (uint32_t base = blockIdx.x * EXPAND_PAIRS; base < n; base += gridDim.x * EXPAND_PAIRS) {
        const uint32_t i = base + (threadIdx.x >> 3);
        bool in = i < n && (coord || nonempty[i]);
        uint32_t x = 0u, y = 0u, z = 0u, cp = 0u;
        if (in) {
            cp = coord ? cptr[i] : i;
            unpack(coord ? coord[i] : 0u, x, y, z);
            /* Parent box in world space: exact integers (tg_sparse_voxel_octree.c:344,359-365). */
            const float pminx = mnx + (float)x * side, pminy = mny + (float)y * side, pminz = mnz + (float)z * side;
            const float pmaxx = pminx + side, pmaxy = pminy + side, pmaxz = pminz + side;
            const float cex = (pmaxx - pminx) * 0.5f, cey = (pmaxy - pminy) * 0.5f, cez = (pmaxz - pminz) * 0.5f;
            const float cminx = pminx + (float)(c % 2) * cex;
            const float cminy = pminy + (float)((c / 2) % 2) * cey;
            const float cminz = pminz + (float)((c / 4) % 2) * cez;
            const float cmaxx = cminx + cex, cmaxy = cminy + cey, cmaxz = cminz + cez;
            const float* m = frames[cp].ws2ms;
            f3 k[8];
            for (int j = 0; j < 8; j++)
                k[j] = mulv(m, (j & 1) ? cmaxx : cminx, (j & 2) ? cmaxy : cminy, (j & 4) ? cmaxz : cminz, 1.0f);
            in = obb_overlaps_cluster(k);
        }
        /* At the root most pairs may have no child at all: where 18 M clusters
         * meet a root of 64^3, a block without one goes on after one barrier
         * instead of three (1.17 -> 1.03 ms, the build 2.45 -> 2.35). */
        if (!coord && !__syncthreads_or(in ? 1 : 0)) continue;
        const uint32_t slot = block_append<EXPAND_BLOCK>(n_out, in ? 1u : 0u);
        if (in) {
            const uint32_t cx = 2u * x + (c & 1u), cy = 2u * y + ((c >> 1) & 1u), cz = 2u * z + (c >> 2);
            if (slot < cap) {
                out_coord[slot] = cx | (cy << 10) | (cz << 20);
                out_cptr[slot] = cp;
            }
        }
        /* a pair's children are one byte of the bitmap */
        const uint32_t kids = (uint32_t)(__ballot(in) >> (threadIdx.x & 56u)) & 0xFFu;
        if (c == 0u && kids) {
            const uint32_t mc = 8u * morton3(x, y, z), v = kids << (mc & 31u);
            if (lds) atomicOr(&s_map[mc >> 5], v);
            else if (v & ~__hip_atomic_load(&map[mc >> 5], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                atomicOr(&map[mc >> 5], v);
        }
        __syncthreads(); /* block_append's shared words and s_map */
    }
    if (lds)
        for (uint32_t w = threadIdx.x; w < map_words; w += EXPAND_BLOCK) {
            const uint32_t v = s_map[w];
            if (v & ~__hip_atomic_load(&map[w], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicOr(&map[w], v);
        }
}

/* Counters and bitmap cleared, but for the root's bit. */
__global__ __launch_bounds__(256) void svo_levels_init_k(uint32_t* __restrict__ cnt, uint32_t n)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) cnt[i] = i == SVO_CNT_N ? 1u : 0u;
}

/* Exclusive scan of count(i), i < n, by one block of 1024 threads that take
 * eight counts each. Returns the total. */
template <typename F>
__device__ static inline uint32_t one_block_scan(uint32_t n, F count, uint32_t* __restrict__ out)
{
    __shared__ uint32_t s_wave[16];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t before = 0u;
    for (uint32_t base = 0; base < n; base += 8192u) {
        const uint32_t i = base + 8u * threadIdx.x;
        const bool full = i + 8u <= n; /* without a test per element the accesses are 16 bytes */
        uint32_t c[8], sum = 0u;
        if (full) {
#pragma unroll
            for (uint32_t k = 0; k < 8u; k++) c[k] = count(i + k);
        } else {
#pragma unroll
            for (uint32_t k = 0; k < 8u; k++) c[k] = i + k < n ? count(i + k) : 0u;
        }
#pragma unroll
        for (uint32_t k = 0; k < 8u; k++) {
            const uint32_t v = c[k];
            c[k] = sum;
            sum += v;
        }
        uint32_t incl = sum;
        for (uint32_t off = 1; off < 64u; off <<= 1) {
            const uint32_t v = __shfl_up(incl, off);
            if (lane >= off) incl += v;
        }
        if (lane == 63u) s_wave[wave] = incl;
        __syncthreads();
        uint32_t total = 0u, mine = before + incl - sum;
        for (uint32_t w = 0; w < 16u; w++) {
            if (w < wave) mine += s_wave[w];
            total += s_wave[w];
        }
        if (full) {
#pragma unroll
            for (uint32_t k = 0; k < 8u; k++) out[i + k] = mine + c[k];
        } else {
#pragma unroll
            for (uint32_t k = 0; k < 8u; k++)
                if (i + k < n) out[i + k] = mine + c[k];
        }
        before += total;
        __syncthreads();
    }
    return before;
}

__global__ __launch_bounds__(256) void svo_popc_k(const uint32_t* __restrict__ map, uint32_t n,
                                                  uint32_t* __restrict__ count)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) count[i] = (uint32_t)__popc(map[i]);
}

/* Numbers the nodes (pre: nodes before each bitmap word, unless scanned
 * already) and tells the host, in its own memory, the pairs and the first node
 * of every level. One block: the 9 k words of depth 11 take it 5 us, where counting, a scan over the chip, the sums and a copy were
 * five launches and 23 us. Beyond SVO_ONE_BLOCK_MAX it is those. */
#define SVO_ONE_BLOCK_MAX 16384u
__global__ __launch_bounds__(1024) void svo_number_k(const uint32_t* __restrict__ cnt, const uint32_t* __restrict__ map,
                                                     uint32_t map_words, uint32_t leaf_level, uint32_t scanned,
                                                     uint32_t* pre, uint32_t* __restrict__ host)
{
    const uint32_t total = scanned ? pre[map_words - 1u] + (uint32_t)__popc(map[map_words - 1u])
                                   : one_block_scan(map_words, [&](uint32_t i) { return (uint32_t)__popc(map[i]); }, pre);
    const uint32_t l = threadIdx.x;
    __threadfence_block();
    __syncthreads();
    if (l > leaf_level + 1u) return;
    host[SVO_CNT_BASE + l] = l <= leaf_level ? pre[node_word(l)] : total;
    host[l] = cnt[l];
}

/* Canonical index of the node of Morton cell m on the level whose bitmap
 * starts at word w0 (its bit must be set). */
__device__ static inline uint32_t node_index(const uint32_t* __restrict__ map, const uint32_t* __restrict__ pre,
                                             uint32_t w0, uint32_t m)
{
    const uint32_t w = w0 + (m >> 5);
    return pre[w] + (uint32_t)__popc(map[w] & ((1u << (m & 31u)) - 1u));
}

/* All nodes from the bitmap, a thread per cell. */
__global__ __launch_bounds__(256) void svo_nodes_k(const uint32_t* __restrict__ map, const uint32_t* __restrict__ pre,
                                                   uint32_t map_words, uint32_t leaf_level, uint32_t leaf_base,
                                                   svo_gnode* __restrict__ nodes, uint32_t* __restrict__ leaf_keys)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x, w = t >> 5;
    if (w >= map_words || !((map[w] >> (t & 31u)) & 1u)) return;
    uint32_t level = 0u, w0 = 0u;
    while (w >= w0 + level_words(level)) w0 += level_words(level++);
    const uint32_t m = t - (w0 << 5);
    const uint32_t idx = node_index(map, pre, w0, m);
    svo_gnode nd;
    nd.first_child = SVO_NONE;
    nd.parent = level ? node_index(map, pre, node_word(level - 1u), m >> 3) : SVO_NONE;
    nd.leaf_idx = SVO_NONE;
    nd.masks = level << 16;
    if (level < leaf_level) {
        const uint32_t w1 = w0 + level_words(level);
        const uint32_t kids = (map[w1 + ((8u * m) >> 5)] >> ((8u * m) & 31u)) & 0xFFu;
        if (kids) {
            nd.first_child = node_index(map, pre, w1, 8u * m + (uint32_t)__ffs((int)kids) - 1u);
            nd.masks |= kids | (level + 1u == leaf_level ? kids << 8 : 0u);
        }
    } else {
        nd.leaf_idx = idx - leaf_base;
        leaf_keys[nd.leaf_idx] = m;
    }
    nd.cx = compact3(m);
    nd.cy = compact3(m >> 1);
    nd.cz = compact3(m >> 2);
    nd.leaf_n = 0;
    nodes[idx] = nd;
}

/* Sort keys of the leaf level's pairs: leaf index << cptr_bits | cluster
 * pointer, so that each leaf's clusters come in pointer order (the
 * reference's list order). */
__global__ __launch_bounds__(256) void svo_pair_keys_k(const uint32_t* __restrict__ coord, const uint32_t* __restrict__ cptr,
                                                       uint32_t n, const uint32_t* __restrict__ map,
                                                       const uint32_t* __restrict__ pre, uint32_t leaf_level,
                                                       uint32_t leaf_base, uint32_t cptr_bits,
                                                       uint64_t* __restrict__ key)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t x, y, z;
    unpack(coord[i], x, y, z);
    const uint32_t leaf = node_index(map, pre, node_word(leaf_level), morton3(x, y, z)) - leaf_base;
    key[i] = ((uint64_t)leaf << cptr_bits) | cptr[i];
}

/* Cluster pointers of the sorted pairs and each leaf's first pair. */
__global__ __launch_bounds__(256) void svo_pair_split_k(const uint64_t* __restrict__ key, uint32_t n, uint32_t cptr_bits,
                                                        uint32_t* __restrict__ cptr, uint32_t* __restrict__ first_pair)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t leaf = (uint32_t)(key[i] >> cptr_bits);
    cptr[i] = (uint32_t)(key[i] & ((1ull << cptr_bits) - 1ull));
    if (i == 0u || (uint32_t)(key[i - 1u] >> cptr_bits) != leaf) first_pair[leaf] = i;
}

/* Notes an exclusive scan whose sums went past 2^32. */
__global__ __launch_bounds__(256) void svo_wrap_k(const uint32_t* __restrict__ count, const uint32_t* __restrict__ off,
                                                  uint32_t n, uint32_t* __restrict__ wrapped)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && off[i] + count[i] < off[i]) *wrapped = 1u;
}

/* Totals of two exclusive scans over n counts, written behind the offsets
 * and to the host's out[0..1]; out[2] to out[4] take the counters
 * SVO_CNT_REUSED, SVO_CNT_MANY and SVO_CNT_WRAP. */
__global__ void svo_totals_k(const uint32_t* __restrict__ count0, uint32_t* __restrict__ off0,
                             const uint32_t* __restrict__ count1, uint32_t* __restrict__ off1, uint32_t n,
                             const uint32_t* __restrict__ cnt, uint32_t* __restrict__ out)
{
    if (threadIdx.x == 2u) out[2] = cnt[SVO_CNT_REUSED];
    if (threadIdx.x == 3u) out[3] = cnt[SVO_CNT_MANY];
    if (threadIdx.x == 4u) out[4] = cnt[SVO_CNT_WRAP];
    if (threadIdx.x > 1u) return;
    const uint32_t* c = threadIdx.x ? count1 : count0;
    uint32_t* o = threadIdx.x ? off1 : off0;
    const uint32_t t = n ? o[n - 1u] + c[n - 1u] : 0u;
    o[n] = t;
    out[threadIdx.x] = t;
}

/* Both scans with their totals in one launch, a block each: 5 us at 3.4 k
 * leaves, against 14 in three launches, which are what longer counts take. Its
 * 2^14 leaves of 2^15 voxels cannot pass 2^32. */
__global__ __launch_bounds__(1024) void svo_offsets_k(const uint32_t* __restrict__ count0, uint32_t* __restrict__ off0,
                                                      const uint32_t* __restrict__ count1, uint32_t* __restrict__ off1,
                                                      uint32_t n, const uint32_t* __restrict__ cnt,
                                                      uint32_t* __restrict__ out)
{
    const uint32_t* c = blockIdx.x ? count1 : count0;
    uint32_t* o = blockIdx.x ? off1 : off0;
    const uint32_t t = one_block_scan(n, [&](uint32_t i) { return c[i]; }, o);
    if (threadIdx.x == 0u) {
        o[n] = t;
        out[blockIdx.x] = t;
        out[2u + blockIdx.x] = cnt[blockIdx.x ? SVO_CNT_MANY : SVO_CNT_REUSED];
        if (blockIdx.x) out[4] = 0u;
    }
}

/* Leaf sampling. A leaf's candidate clusters are staged LEAF_STAGE at a time:
 * eight lanes per cluster transform its corners (the cluster's in world space
 * for the trimmed voxel range, the block's in cluster space for the
 * interpolation), and its solid bits go to LDS. The waves of the workgroup then
 * take clusters in turn, a lane per (y, z) row of the range: the interpolation
 * over z and y is done once per row and only the one over x per voxel, in the
 * reference's operation order (tg_sparse_voxel_octree.c:242-291), and a row's
 * samples are the bits of one word of the leaf.
 *
 * Bound by the samples' arithmetic: a cluster covers about 14^3 voxels of its
 * leaf. One voxel per lane with the full interpolation took 80 instructions a
 * sample and two barriers a cluster; now about 30 and none, so that waves run
 * different clusters at once and the leaf with the most clusters (164 of 16 on
 * average) no longer makes the launch. 512 objects, depth 11: bits 0.69 -> 0.16
 * ms, materials 0.73 -> 0.29 ms. 512 lanes against 256: 0.16 and 0.20 ms. */
#define LEAF_BLOCK 512u
/* A launch holds less than 2^32 lanes along a dimension, and takes more modulo
 * 2^32 without an error: the leaves' workgroups lie in rows of LEAF_ROW leaves. */
#define LEAF_ROW (1u << 18)
/* Bits: a leaf of few candidates leaves most of 512 lanes idle and is one chain
 * of dependent loads, so where the leaves have up to LEAF_SPARSE candidates on
 * average their workgroups are of LEAF_SPARSE_BLOCK lanes, four times as many at
 * once. 200 thousand single clusters in 267 thousand leaves: 512 lanes 3.29 ms,
 * 256 1.19, 128 0.81; 5000 objects of up to 27 clusters 0.23, 0.13, 0.14. From
 * five to eight on average the two are equal (0.31 ms), below two 128 lanes are
 * needed (0.46 against 0.17). */
#define LEAF_SPARSE 4u
#define LEAF_SPARSE_BLOCK 128u
/* Materials: leaves of up to LEAF_FEW candidates and LEAF_FEW_SOLID solid
 * voxels are svo_leaf_mats_few_k's, a workgroup each; the others are
 * svo_leaf_mats_k's, whose four workgroups clear and read 32768 keys whatever
 * the leaf holds. 267 thousand leaves of one or two clusters: 10.8 ms there, 1.01
 * here (2.50 with a limit of 512 voxels); 14 thousand of seven 0.79 and 0.47. The
 * limits of 8, 16 and 32 candidates measure the same; beyond 2048 voxels 256
 * lanes take longer than 2048 (646 leaves, limit 4096: 113 us against 71), and
 * fewer than LEAF_FEW_LEAVES leaves do not fill the chip with one workgroup each
 * (86 against 71). svo_leaf_k lists the others: with a launch over all leaves that
 * returned for the few, one dense leaf among 449 thousand cost 1.7 ms. */
#define LEAF_FEW 16u
#define LEAF_FEW_SOLID 2048u
#define LEAF_FEW_LEAVES 1024u

__device__ static inline bool leaf_few(uint32_t candidates, uint32_t solid, uint32_t few)
{
    return candidates <= few && solid <= LEAF_FEW_SOLID;
}

/* Candidate clusters of a workgroup of kBlock lanes. */
template <uint32_t kBlock>
struct leaf_stage {
    static constexpr uint32_t kCount = kBlock / 8u;
    float    c[kCount][24];          /* block corners in cluster space, x y z each */
    uint32_t lo[kCount];             /* trimmed range: x | y << 8 | z << 16 ... */
    uint32_t hi[kCount];             /* ... one past it; equal where empty */
    uint32_t cidx[kCount];
    uint32_t lut[kCount];
    uint32_t bits[kCount][16];
};

/* Stages n clusters from pair_cptr; slices z0 .. z1 of the leaf only. */
template <uint32_t kBlock>
__device__ static inline void leaf_stage_load(leaf_stage<kBlock>& st, const uint32_t* __restrict__ pair_cptr, uint32_t n,
                                              const svo_frame* __restrict__ frames, const uint32_t* __restrict__ bits,
                                              float pminx, float pminy, float pminz, uint32_t quirk, uint32_t z0,
                                              uint32_t z1)
{
    const uint32_t k = threadIdx.x >> 3, i = threadIdx.x & 7u;
    const float pmaxx = pminx + 32.0f, pmaxy = pminy + 32.0f, pmaxz = pminz + 32.0f;
    if (k < n) {
        const svo_frame& f = frames[pair_cptr[k]];
        const f3 bc = mulv(f.ws2cs, (i & 1u) ? pmaxx : pminx, (i & 2u) ? pmaxy : pminy, (i & 4u) ? pmaxz : pminz, 1.0f);
        st.c[k][3u * i] = bc.x; st.c[k][3u * i + 1u] = bc.y; st.c[k][3u * i + 2u] = bc.z;
        /* the cluster's AABB over its corners (:134-197); the reductions pair
         * corners as the reference's min / max expressions nest, (0 1) (2 3)
         * (4 6) (5 7), with corner 2 again in place of 3 under the quirk */
        const f3 cw = mulv(f.cs2ws, (i & 1u) ? 8.0f : 0.0f, (i & 2u) ? 8.0f : 0.0f, (i & 4u) ? 8.0f : 0.0f, 1.0f);
        f3 mn = cw, mx = cw;
        const uint32_t lane = threadIdx.x & 63u, g = lane & ~7u;
        const uint32_t p1 = i == 4u ? 6u : i == 5u ? 7u : i == 2u ? (quirk ? 2u : 3u) : i == 0u ? 1u : i;
        const uint32_t p2 = i == 0u ? 2u : i == 4u ? 5u : i, p3 = i == 0u ? 4u : i;
        const uint32_t part[3] = {g | p1, g | p2, g | p3};
#pragma unroll
        for (int r = 0; r < 3; r++) {
            const f3 on = {__shfl(mn.x, (int)part[r]), __shfl(mn.y, (int)part[r]), __shfl(mn.z, (int)part[r])};
            const f3 ox = {__shfl(mx.x, (int)part[r]), __shfl(mx.y, (int)part[r]), __shfl(mx.z, (int)part[r])};
            mn = {fmin2(mn.x, on.x), fmin2(mn.y, on.y), fmin2(mn.z, on.z)};
            mx = {fmax2(mx.x, ox.x), fmax2(mx.y, ox.y), fmax2(mx.z, ox.z)};
        }
        if (i == 0u) {
            /* trimmed box (:218-233), clamped into [0, 32] */
            const float tlo[3] = {fmax2(pminx, floorf(mn.x)) - pminx, fmax2(pminy, floorf(mn.y)) - pminy, fmax2(pminz, floorf(mn.z)) - pminz};
            const float thi[3] = {fmin2(pmaxx, ceilf(mx.x)) - pminx, fmin2(pmaxy, ceilf(mx.y)) - pminy, fmin2(pmaxz, ceilf(mx.z)) - pminz};
            uint32_t lo[3], hi[3];
            for (int a = 0; a < 3; a++) {
                lo[a] = (uint32_t)fmin2(32.0f, fmax2(0.0f, tlo[a]));
                hi[a] = (uint32_t)fmin2(32.0f, fmax2(0.0f, thi[a]));
            }
            lo[2] = lo[2] > z0 ? lo[2] : z0;
            hi[2] = hi[2] < z1 ? hi[2] : z1;
            const bool empty = hi[0] <= lo[0] || hi[1] <= lo[1] || hi[2] <= lo[2];
            st.lo[k] = lo[0] | (lo[1] << 8) | (lo[2] << 16);
            st.hi[k] = empty ? st.lo[k] : hi[0] | (hi[1] << 8) | (hi[2] << 16);
            st.cidx[k] = f.cidx;
            st.lut[k] = f.lut;
        }
    }
    for (uint32_t j = threadIdx.x; j < 16u * n; j += kBlock)
        st.bits[j >> 4][j & 15u] = bits[(size_t)frames[pair_cptr[j >> 4]].cidx * 16u + (j & 15u)];
}

/* Ends of row (y, z) in cluster space, interpolated over z, then y. */
__device__ static inline void leaf_row_ends(const float* c, uint32_t y, uint32_t z, float p0[3], float p1[3])
{
    const float tz = ((float)z + 0.5f) / 32.0f, omtz = 1.0f - tz;
    const float ty = ((float)y + 0.5f) / 32.0f, omty = 1.0f - ty;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const float pz0 = omtz * c[a] + tz * c[12 + a], pz1 = omtz * c[3 + a] + tz * c[15 + a];
        const float pz2 = omtz * c[6 + a] + tz * c[18 + a], pz3 = omtz * c[9 + a] + tz * c[21 + a];
        p0[a] = omty * pz0 + ty * pz2;
        p1[a] = omty * pz1 + ty * pz3;
    }
}

/* The cluster voxel v that the row's sample x falls on; false for none. */
__device__ static inline bool leaf_voxel(const float p0[3], const float p1[3], uint32_t x, uint32_t& v)
{
    const float tx = ((float)x + 0.5f) / 32.0f, omtx = 1.0f - tx;
    /* 0 <= centre < 8 on each axis as its floor in 0 .. 7 */
    const uint32_t ix = (uint32_t)(int)floorf(omtx * p0[0] + tx * p1[0]);
    const uint32_t iy = (uint32_t)(int)floorf(omtx * p0[1] + tx * p1[1]);
    const uint32_t iz = (uint32_t)(int)floorf(omtx * p0[2] + tx * p1[2]);
    v = 64u * iz + 8u * iy + ix;
    return (ix | iy | iz) < 8u;
}

/* Calls f(row word 32 z + y of the leaf, voxel x, cluster voxel v) for every
 * sample of staged cluster k that falls on a solid voxel, a lane per row;
 * row_done(row word) after each row. Called by whole waves. */
template <uint32_t kBlock, typename F, typename R>
__device__ static inline void leaf_rows(const leaf_stage<kBlock>& st, uint32_t k, F&& f, R&& row_done)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t lo = __builtin_amdgcn_readfirstlane(st.lo[k]), hi = __builtin_amdgcn_readfirstlane(st.hi[k]);
    if (lo == hi) return;
    const uint32_t x0 = lo & 255u, y0 = (lo >> 8) & 255u, z0 = lo >> 16;
    const uint32_t x1 = hi & 255u, ny = ((hi >> 8) & 255u) - y0, n_rows = ny * ((hi >> 16) - z0);
    const uint32_t inv = 65536u / ny + 1u;   /* r / ny for r < 1024, ny <= 32 */
    const float* c = st.c[k];
    for (uint32_t r = lane; r < n_rows; r += 64u) {
        const uint32_t q = (r * inv) >> 16;
        const uint32_t y = y0 + r - q * ny, z = z0 + q;
        float p0[3], p1[3];
        leaf_row_ends(c, y, z, p0, p1);
        for (uint32_t x = x0; x < x1; x++) {
            uint32_t v;
            if (leaf_voxel(p0, p1, x, v) && ((st.bits[k][v >> 5] >> (v & 31u)) & 1u)) f(x, v, 32u * z + y);
        }
        row_done(32u * z + y);
    }
}

/* First pass, a workgroup per leaf: its bits, the per-word prefix counts that
 * index its materials (wpre[w] = solid voxels in the leaf's words before w),
 * its solid voxel count and its list: the clusters with a sample on a solid
 * voxel, in candidate order. */
template <uint32_t kBlock>
__global__ __launch_bounds__(kBlock) void svo_leaf_k(const svo_gnode* __restrict__ nodes, uint32_t leaf_base,
                                                         const uint32_t* __restrict__ pair_cptr,
                                                         const uint32_t* __restrict__ leaf_first_pair, uint32_t n_pairs,
                                                         uint32_t n_leaves, const svo_frame* __restrict__ frames,
                                                         const uint32_t* __restrict__ bits, float mnx, float mny,
                                                         float mnz, uint32_t quirk, uint32_t* __restrict__ leaf_bits,
                                                         uint32_t* __restrict__ leaf_solid, uint16_t* __restrict__ wpre,
                                                         uint32_t* __restrict__ leaf_n, uint32_t* __restrict__ list_tmp,
                                                         svo_gnode* __restrict__ nodes_rw,
                                                         const uint32_t* __restrict__ reuse,
                                                         const uint32_t* __restrict__ old_bits,
                                                         const uint32_t* __restrict__ old_off,
                                                         const uint16_t* __restrict__ old_wpre,
                                                         const uint32_t* __restrict__ old_n,
                                                         const uint32_t* __restrict__ old_list_off,
                                                         const uint32_t* __restrict__ old_list,
                                                         uint32_t few, uint32_t* __restrict__ n_many,
                                                         uint32_t* __restrict__ many)
{
    constexpr uint32_t kStage = leaf_stage<kBlock>::kCount;
    const uint32_t leaf = blockIdx.y * gridDim.x + blockIdx.x, tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    if (leaf >= n_leaves) return;
    const uint32_t b = leaf_first_pair[leaf];
    const uint32_t e = leaf + 1 < n_leaves ? leaf_first_pair[leaf + 1] : n_pairs;
    if (reuse && reuse[leaf] != SVO_NONE) {
        /* an update: same candidate clusters in the same order, none of
         * them new, so the previous build's leaf is this leaf */
        const uint32_t j = reuse[leaf];
        const uint4* sb = (const uint4*)(old_bits + (size_t)j * TGX_SVO_BLOCK_WORDS);
        uint4* db = (uint4*)(leaf_bits + (size_t)leaf * TGX_SVO_BLOCK_WORDS);
        const uint2* sw = (const uint2*)(old_wpre + (size_t)j * TGX_SVO_BLOCK_WORDS);
        uint2* dw = (uint2*)(wpre + (size_t)leaf * TGX_SVO_BLOCK_WORDS);
        for (uint32_t w = tid; w < TGX_SVO_BLOCK_WORDS / 4u; w += kBlock) {
            db[w] = sb[w];
            dw[w] = sw[w];
        }
        const uint32_t n = old_n[j], o = old_list_off[j];
        for (uint32_t i = tid; i < n; i += kBlock) list_tmp[b + i] = old_list[o + i];
        if (tid == 0) {
            leaf_n[leaf] = n;
            nodes_rw[leaf_base + leaf].leaf_n = n;
            const uint32_t solid = old_off[j + 1] - old_off[j];
            leaf_solid[leaf] = solid;
            if (few && !leaf_few(e - b, solid, few)) many[atomicAdd(n_many, 1u)] = leaf;
        }
        return;
    }
    __shared__ leaf_stage<kBlock> st;
    __shared__ uint32_t lbits[TGX_SVO_BLOCK_WORDS];
    __shared__ uint32_t s_any[kStage];
    __shared__ uint32_t wsum[kBlock / 64u];
    const svo_gnode nd = nodes[leaf_base + leaf];
    const float pminx = mnx + (float)nd.cx * 32.0f, pminy = mny + (float)nd.cy * 32.0f, pminz = mnz + (float)nd.cz * 32.0f;
    for (uint32_t w = tid; w < TGX_SVO_BLOCK_WORDS; w += kBlock) lbits[w] = 0u;
    /* wave 0: list entries so far, and the last flagged cluster */
    uint32_t n_contrib = 0u, last_cidx = SVO_NONE;
    for (uint32_t s0 = b; s0 < e; s0 += kStage) {
        const uint32_t n = e - s0 < kStage ? e - s0 : kStage;
        leaf_stage_load(st, pair_cptr + s0, n, frames, bits, pminx, pminy, pminz, quirk, 0u, 32u);
        __syncthreads();
        for (uint32_t k = wave; k < n; k += kBlock / 64u) {
            uint32_t mask = 0u, any = 0u;
            leaf_rows(st, k, [&](uint32_t x, uint32_t, uint32_t) { mask |= 1u << x; },
                      [&](uint32_t w) {
                          if (mask) atomicOr(&lbits[w], mask);
                          any |= mask;
                          mask = 0u;
                      });
            const bool some = __any(any != 0u);
            if (lane == 0u) s_any[k] = some ? 1u : 0u;
        }
        __syncthreads();
        if (wave == 0u) {
            /* the flagged clusters in order; one equal to the flagged
             * cluster before it is listed once */
            const bool flag = lane < n && s_any[lane] != 0u;
            const uint32_t c = lane < n ? st.cidx[lane] : SVO_NONE;
            const unsigned long long fm = __ballot(flag);
            const unsigned long long below = fm & ((1ull << lane) - 1ull);
            const uint32_t prev = __shfl(c, below ? 63 - __clzll((long long)below) : 0);
            const bool keep = flag && c != (below ? prev : last_cidx);
            const unsigned long long km = __ballot(keep);
            if (keep) list_tmp[b + n_contrib + (uint32_t)__popcll(km & ((1ull << lane) - 1ull))] = c;
            n_contrib += (uint32_t)__popcll(km);
            if (fm) last_cidx = __shfl(c, 63 - __clzll((long long)fm));
        }
        /* st is rewritten by the next stage */
        __syncthreads();
    }
    __syncthreads();
    /* bits, prefix counts and total: kWords words per thread */
    constexpr uint32_t kWords = TGX_SVO_BLOCK_WORDS / kBlock;
    uint32_t w[kWords], pre[kWords], cnt = 0u;
#pragma unroll
    for (uint32_t k = 0; k < kWords; k++) {
        w[k] = lbits[kWords * tid + k];
        pre[k] = cnt;
        cnt += (uint32_t)__popc(w[k]);
    }
    uint32_t incl = cnt;
#pragma unroll
    for (uint32_t d = 1; d < 64u; d <<= 1) {
        const uint32_t u = __shfl_up(incl, d);
        if (lane >= d) incl += u;
    }
    if (lane == 63u) wsum[wave] = incl;
    __syncthreads();
    uint32_t run = incl - cnt, total = 0u;
    for (uint32_t k = 0; k < kBlock / 64u; k++) {
        run += k < wave ? wsum[k] : 0u;
        total += wsum[k];
    }
    uint32_t* gb = leaf_bits + (size_t)leaf * TGX_SVO_BLOCK_WORDS + kWords * tid;
    uint32_t* gp = (uint32_t*)(wpre + (size_t)leaf * TGX_SVO_BLOCK_WORDS) + kWords / 2u * tid;
#pragma unroll
    for (uint32_t k = 0; k < kWords; k++) gb[k] = w[k];
#pragma unroll
    for (uint32_t k = 0; k < kWords / 2u; k++) gp[k] = (run + pre[2u * k]) | ((run + pre[2u * k + 1u]) << 16);
    if (tid == 0) {
        leaf_n[leaf] = n_contrib;
        nodes_rw[leaf_base + leaf].leaf_n = n_contrib;
        leaf_solid[leaf] = total;
        if (few && !leaf_few(e - b, total, few)) many[atomicAdd(n_many, 1u)] = leaf;
    }
}

/* Second pass (after the counts are scanned into mat_off) for all leaves but
 * those of few candidates (leaf_few), LEAF_PARTS workgroups per leaf, eight z
 * slices each: the materials of the leaf's solid voxels, in bit order, at
 * mat_off[leaf] in the pool. A voxel's material is
 * that of the first candidate that samples it solid: the samples of a
 * candidate k on cluster voxel v lower the voxel's key to k << 9 | v, so waves
 * run different candidates in any order (a wave's lanes are on rows of the
 * same x: each row's keys are rotated by exclusive or so that they fall on
 * different LDS banks: 0.38 -> 0.29 ms). One workgroup a leaf holds 128 KB of
 * keys and takes 0.54 ms, 2, 4 and 8 take 0.35, 0.29 and 0.45. Keys hold 2^LEAF_SPAN candidates;
 * more are taken in turns, each turn filling voxels that no earlier one has. */
#define LEAF_PARTS 4u
#define LEAF_SLICES (32u / LEAF_PARTS)
#define LEAF_SPAN 22u
__global__ __launch_bounds__(LEAF_BLOCK) void svo_leaf_mats_k(const svo_gnode* __restrict__ nodes, uint32_t leaf_base,
                                                              const uint32_t* __restrict__ pair_cptr,
                                                              const uint32_t* __restrict__ leaf_first_pair,
                                                              uint32_t n_pairs, uint32_t n_leaves,
                                                              const svo_frame* __restrict__ frames,
                                                              const uint32_t* __restrict__ bits,
                                                              const uint8_t* __restrict__ materials, float mnx,
                                                              float mny, float mnz, uint32_t quirk,
                                                              const uint32_t* __restrict__ leaf_bits,
                                                              const uint16_t* __restrict__ wpre,
                                                              const uint32_t* __restrict__ mat_off,
                                                              uint16_t* __restrict__ pool,
                                                              const uint32_t* __restrict__ reuse,
                                                              const uint32_t* __restrict__ old_off,
                                                              const uint16_t* __restrict__ old_pool,
                                                              const uint32_t* __restrict__ many, uint32_t n_many)
{
    const uint32_t i_many = blockIdx.y * (gridDim.x / LEAF_PARTS) + blockIdx.x / LEAF_PARTS, part = blockIdx.x % LEAF_PARTS;
    const uint32_t tid = threadIdx.x, wave = tid >> 6;
    if (i_many >= n_many) return;
    const uint32_t leaf = many ? many[i_many] : i_many; /* null: all leaves */
    const uint32_t b = leaf_first_pair[leaf];
    const uint32_t e = leaf + 1 < n_leaves ? leaf_first_pair[leaf + 1] : n_pairs;
    if (reuse && reuse[leaf] != SVO_NONE) {
        const uint32_t j = reuse[leaf];
        const uint32_t o = old_off[j], n = old_off[j + 1] - o, d = mat_off[leaf];
        for (uint32_t i = part * LEAF_BLOCK + tid; i < n; i += LEAF_PARTS * LEAF_BLOCK) pool[d + i] = old_pool[o + i];
        return;
    }
    constexpr uint32_t kStage = leaf_stage<LEAF_BLOCK>::kCount;
    __shared__ leaf_stage<LEAF_BLOCK> st;
    __shared__ uint32_t key[LEAF_SLICES * 1024u];
    __shared__ uint32_t s_bits[LEAF_SLICES * 32u], s_done[LEAF_SLICES * 32u];
    const svo_gnode nd = nodes[leaf_base + leaf];
    const float pminx = mnx + (float)nd.cx * 32.0f, pminy = mny + (float)nd.cy * 32.0f, pminz = mnz + (float)nd.cz * 32.0f;
    const uint32_t z0 = part * LEAF_SLICES, row0 = 32u * z0;
    const size_t word0 = (size_t)leaf * TGX_SVO_BLOCK_WORDS + row0;
    for (uint32_t w = tid; w < LEAF_SLICES * 32u; w += LEAF_BLOCK) {
        s_bits[w] = leaf_bits[word0 + w];
        s_done[w] = 0u;
    }
    uint16_t* mats = pool + mat_off[leaf];
    for (uint32_t t0 = b; t0 < e; t0 += 1u << LEAF_SPAN) {
        const uint32_t t1 = e - t0 < (1u << LEAF_SPAN) ? e : t0 + (1u << LEAF_SPAN);
        for (uint32_t v = tid; v < LEAF_SLICES * 1024u; v += LEAF_BLOCK) key[v] = SVO_NONE;
        for (uint32_t s0 = t0; s0 < t1; s0 += kStage) {
            const uint32_t n = t1 - s0 < kStage ? t1 - s0 : kStage;
            leaf_stage_load(st, pair_cptr + s0, n, frames, bits, pminx, pminy, pminz, quirk, z0, z0 + LEAF_SLICES);
            __syncthreads();
            for (uint32_t k = wave; k < n; k += LEAF_BLOCK / 64u)
                leaf_rows(st, k,
                          [&](uint32_t x, uint32_t v, uint32_t w) {
                              atomicMin(&key[32u * (w - row0) + (x ^ (w & 31u))], ((s0 - t0 + k) << 9) | v);
                          },
                          [](uint32_t) {});
            /* st is rewritten by the next stage */
            __syncthreads();
        }
        /* a half wave per row */
        for (uint32_t i = tid; i < LEAF_SLICES * 1024u; i += LEAF_BLOCK) {
            const uint32_t w = i >> 5, m = 1u << (i & 31u), q = key[i ^ (w & 31u)];
            const bool mine = q != SVO_NONE && !(s_done[w] & m);
            if (mine) {
                const svo_frame& f = frames[pair_cptr[t0 + (q >> 9)]];
                mats[(uint32_t)wpre[word0 + w] + (uint32_t)__popc(s_bits[w] & (m - 1u))] =
                    (uint16_t)(f.lut | (materials ? (uint32_t)materials[(size_t)f.cidx * TGX_VOXELS_PER_CLUSTER + (q & 511u)] : 0u));
            }
            /* rows are 32 consecutive lanes: the half wave's ballot */
            const unsigned long long got = __ballot(mine);
            if ((i & 31u) == 0u) s_done[w] |= (uint32_t)(got >> (tid & 32u));
        }
        __syncthreads();
    }
}

/* The same for the leaves of leaf_few, a workgroup per leaf and a lane per solid
 * voxel in the pool's order: it looks its voxel up in the leaf's prefix counts
 * and samples it for the candidates in turn until one has it solid (the first
 * pass found one). Bound by its chain of loads, eight workgroups a CU. */
#define LEAF_FEW_BLOCK 256u
__global__ __launch_bounds__(LEAF_FEW_BLOCK) void svo_leaf_mats_few_k(
    const svo_gnode* __restrict__ nodes, uint32_t leaf_base, const uint32_t* __restrict__ pair_cptr,
    const uint32_t* __restrict__ leaf_first_pair, uint32_t n_pairs, uint32_t n_leaves,
    const svo_frame* __restrict__ frames, const uint32_t* __restrict__ bits, const uint8_t* __restrict__ materials,
    float mnx, float mny, float mnz, uint32_t quirk, const uint32_t* __restrict__ leaf_bits,
    const uint16_t* __restrict__ wpre, const uint32_t* __restrict__ mat_off, uint16_t* __restrict__ pool,
    const uint32_t* __restrict__ reuse, const uint32_t* __restrict__ old_off, const uint16_t* __restrict__ old_pool,
    const uint32_t* __restrict__, uint32_t few)
{
    const uint32_t leaf = blockIdx.y * gridDim.x + blockIdx.x, tid = threadIdx.x;
    if (leaf >= n_leaves) return;
    const uint32_t b = leaf_first_pair[leaf];
    const uint32_t e = leaf + 1 < n_leaves ? leaf_first_pair[leaf + 1] : n_pairs;
    const uint32_t n = e - b, off = mat_off[leaf], n_solid = mat_off[leaf + 1] - off;
    if (!leaf_few(n, n_solid, few)) return;
    uint16_t* mats = pool + off;
    if (reuse && reuse[leaf] != SVO_NONE) {
        const uint16_t* old = old_pool + old_off[reuse[leaf]];
        for (uint32_t i = tid; i < n_solid; i += LEAF_FEW_BLOCK) mats[i] = old[i];
        return;
    }
    static_assert(LEAF_FEW <= leaf_stage<LEAF_FEW_BLOCK>::kCount, "one stage holds the candidates");
    __shared__ leaf_stage<LEAF_FEW_BLOCK> st;
    __shared__ uint32_t s_bits[TGX_SVO_BLOCK_WORDS];
    __shared__ uint16_t s_pre[TGX_SVO_BLOCK_WORDS];
    const svo_gnode nd = nodes[leaf_base + leaf];
    const float pminx = mnx + (float)nd.cx * 32.0f, pminy = mny + (float)nd.cy * 32.0f, pminz = mnz + (float)nd.cz * 32.0f;
    const size_t word0 = (size_t)leaf * TGX_SVO_BLOCK_WORDS;
    for (uint32_t w = tid; w < TGX_SVO_BLOCK_WORDS; w += LEAF_FEW_BLOCK) {
        s_bits[w] = leaf_bits[word0 + w];
        s_pre[w] = wpre[word0 + w];
    }
    leaf_stage_load(st, pair_cptr + b, n, frames, bits, pminx, pminy, pminz, quirk, 0u, 32u);
    __syncthreads();
    for (uint32_t i = tid; i < n_solid; i += LEAF_FEW_BLOCK) {
        /* the last word with a prefix count of up to i, and its bit */
        uint32_t w = 0u;
        for (uint32_t s = TGX_SVO_BLOCK_WORDS / 2u; s; s >>= 1)
            if (s_pre[w + s] <= i) w += s;
        uint32_t m = s_bits[w], r = i - s_pre[w], x = 0u;
#pragma unroll
        for (uint32_t s = 16u; s; s >>= 1) {
            const uint32_t c = (uint32_t)__popc(m & ((1u << s) - 1u));
            const bool up = r >= c;
            r -= up ? c : 0u;
            x += up ? s : 0u;
            m = up ? m >> s : m;
        }
        const uint32_t y = w & 31u, z = w >> 5;
        for (uint32_t k = 0; k < n; k++) {
            const uint32_t lo = st.lo[k], hi = st.hi[k];
            if (lo == hi || x < (lo & 255u) || x >= (hi & 255u) || y < ((lo >> 8) & 255u) || y >= ((hi >> 8) & 255u) ||
                z < lo >> 16 || z >= hi >> 16)
                continue;
            float p0[3], p1[3];
            leaf_row_ends(st.c[k], y, z, p0, p1);
            uint32_t v;
            if (!leaf_voxel(p0, p1, x, v) || !((st.bits[k][v >> 5] >> (v & 31u)) & 1u)) continue;
            mats[i] = (uint16_t)(st.lut[k] |
                                 (materials ? (uint32_t)materials[(size_t)st.cidx[k] * TGX_VOXELS_PER_CLUSTER + v] : 0u));
            break;
        }
    }
}

/* Update: for each new leaf, the previous build's leaf with the same key
 * whose candidate clusters (cluster indices in pointer order) are the same
 * and none of them placed since that build; SVO_NONE otherwise. */
__global__ __launch_bounds__(256) void svo_match_k(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ first,
                                                   uint32_t n_pairs, uint32_t n_leaves,
                                                   const uint32_t* __restrict__ pair_cptr,
                                                   const svo_frame* __restrict__ frames, const uint8_t* __restrict__ dirty,
                                                   const uint32_t* __restrict__ prev_keys, uint32_t n_prev,
                                                   const uint32_t* __restrict__ prev_off,
                                                   const uint32_t* __restrict__ prev_cand, uint32_t* __restrict__ reuse,
                                                   uint32_t* __restrict__ n_reused)
{
    /* one wave per leaf: the search is wave-uniform, the candidates are
     * compared 64 at a time */
    const uint32_t l = blockIdx.x * (blockDim.x / 64u) + threadIdx.x / 64u;
    const uint32_t lane = threadIdx.x & 63u;
    if (l >= n_leaves) return;
    const uint32_t key = keys[l];
    uint32_t lo = 0, hi = n_prev;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (prev_keys[mid] < key) lo = mid + 1; else hi = mid;
    }
    uint32_t r = SVO_NONE;
    if (lo < n_prev && prev_keys[lo] == key) {
        const uint32_t b = first[l], e = l + 1 < n_leaves ? first[l + 1] : n_pairs;
        const uint32_t pb = prev_off[lo], pe = prev_off[lo + 1];
        if (e - b == pe - pb) {
            uint32_t bad = 0u;
            for (uint32_t k = lane; k < e - b; k += 64u) {
                const uint32_t c = frames[pair_cptr[b + k]].cidx;
                bad |= (c != prev_cand[pb + k] || dirty[c] != 0u) ? 1u : 0u;
            }
            if (__ballot(bad != 0u) == 0ull) r = lo;
        }
    }
    if (lane == 0) {
        reuse[l] = r;
        if (r != SVO_NONE) atomicAdd(n_reused, 1u);
    }
}

/* What the next update compares against: leaf keys, first pairs, candidate
 * cluster indices; and no cluster is dirty any more. */
__global__ __launch_bounds__(256) void svo_keep_k(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ first,
                                                  uint32_t n_leaves, const uint32_t* __restrict__ pair_cptr,
                                                  uint32_t n_pairs, const svo_frame* __restrict__ frames,
                                                  uint32_t dirty_words, uint32_t* __restrict__ prev_keys,
                                                  uint32_t* __restrict__ prev_off, uint32_t* __restrict__ prev_cand,
                                                  uint32_t* __restrict__ dirty)
{
    const uint64_t step = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;; i += step) {
        if (i < n_leaves) prev_keys[i] = keys[i];
        if (i <= n_leaves) prev_off[i] = i < n_leaves ? first[i] : n_pairs;
        if (i < n_pairs) prev_cand[i] = frames[pair_cptr[i]].cidx;
        if (i < dirty_words) dirty[i] = 0u;
        if (i >= n_leaves && i >= n_pairs && i >= dirty_words) return;
    }
}

/* A wave per leaf: one bit per 8^3 brick (bx + 4 by + 16 bz, a lane each) that
 * holds a solid voxel; and with list_tmp the leaf's list from its first
 * pair's place to its offset. */
__global__ __launch_bounds__(256) void svo_bricks_k(const uint32_t* __restrict__ leaf_bits, uint32_t n_leaves,
                                                    unsigned long long* __restrict__ bricks,
                                                    const uint32_t* __restrict__ list_tmp,
                                                    const uint32_t* __restrict__ first_pair,
                                                    const uint32_t* __restrict__ leaf_n,
                                                    const uint32_t* __restrict__ list_off, uint32_t* __restrict__ list)
{
    const uint32_t l = blockIdx.x * 4u + (threadIdx.x >> 6), t = threadIdx.x & 63u;
    if (l >= n_leaves) return;
    const uint32_t bx = t & 3u, by = (t >> 2) & 3u, bz = t >> 4;
    const uint32_t* g = leaf_bits + (size_t)l * TGX_SVO_BLOCK_WORDS;
    uint32_t acc = 0;
    for (uint32_t z = 8u * bz; z < 8u * bz + 8u; z++)
        for (uint32_t y = 8u * by; y < 8u * by + 8u; y++) acc |= (g[32u * z + y] >> (8u * bx)) & 0xFFu;
    const unsigned long long m = __ballot(acc != 0u);
    if (t == 0) bricks[l] = m;
    if (!list_tmp) return;
    const uint32_t b = first_pair[l], o = list_off[l], n = leaf_n[l];
    for (uint32_t i = t; i < n; i += 64u) list[o + i] = list_tmp[b + i];
}

/* Leaf grid for traversal, one entry per 32^3 cell of the root (cell x | y
 * << leaf_level | z << 2 leaf_level): the leaf's index, or for a cell without
 * a leaf that holds solid voxels SVO_GRID_EMPTY | q, the child slot that the
 * descent to the cell ends in being 2^q cells wide. 1 MB at depth 11, 8 MB at
 * 12, 64 MB at 13. A thread per 2^3 cells, one descent to the node that holds
 * them and four stores: bound by those (15 us at depth 13, 4.4 TB/s; a descent
 * per cell took 34). */
__global__ __launch_bounds__(256) void svo_grid_k(const svo_gnode* __restrict__ nodes, uint32_t leaf_level,
                                                  const unsigned long long* __restrict__ bricks,
                                                  uint32_t* __restrict__ grid)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t l = leaf_level - 1u, m = (1u << l) - 1u;
    if (i >> (3u * l)) return;
    const uint32_t x = i & m, y = (i >> l) & m, z = i >> (2u * l);
    uint32_t node = 0u, empty = SVO_GRID_EMPTY, valid = nodes[0].masks & 0xFFu;
    for (uint32_t q = l; q-- > 0u;) {
        const uint32_t rc = ((x >> q) & 1u) | (((y >> q) & 1u) << 1) | (((z >> q) & 1u) << 2);
        if (!(valid & (1u << rc))) {
            empty = SVO_GRID_EMPTY | (q + 1u);
            valid = 0u;
            break;
        }
        node = nodes[node].first_child + (uint32_t)__popc(valid & ((1u << rc) - 1u));
        valid = nodes[node].masks & 0xFFu;
    }
    uint32_t cell[8], child = valid ? nodes[node].first_child : 0u;
#pragma unroll
    for (uint32_t rc = 0; rc < 8u; rc++) {
        cell[rc] = empty;
        if (valid & (1u << rc)) {
            const uint32_t leaf = nodes[child++].leaf_idx;
            cell[rc] = bricks[leaf] ? leaf : SVO_GRID_EMPTY;
        }
    }
#pragma unroll
    for (uint32_t r = 0; r < 4u; r++)
        *(uint2*)&grid[2u * x + ((2u * y + (r & 1u)) << leaf_level) + ((2u * z + (r >> 1)) << (2u * leaf_level))] =
            make_uint2(cell[2u * r], cell[2u * r + 1u]);
}

/* ------------------------------------------------------------------------ */
/* Host side                                                                */
/* ------------------------------------------------------------------------ */

void tgx_svo_release(tgx_context* ctx)
{
    tgx_buffer* bufs[] = {&ctx->svo_nodes, &ctx->svo_leaf_bits, &ctx->svo_leaf_mats, &ctx->svo_leaf_moff,
                          &ctx->svo_leaf_wpre, &ctx->svo_old_moff, &ctx->svo_old_wpre, &ctx->svo_leaf_n,
                          &ctx->svo_list_off, &ctx->svo_list, &ctx->svo_frames, &ctx->svo_rays,
                          &ctx->svo_hits, &ctx->prim_tmp, &ctx->gi_counts, &ctx->gi_surf,
                          &ctx->gi_rays, &ctx->gi_res, &ctx->gi_shadow, &ctx->gi_shadow_res,
                          &ctx->gi_weight, &ctx->gi_contrib, &ctx->gi_list, &ctx->gi_rays2, &ctx->gi_sort, &ctx->gi_bsurf, &ctx->gi_blist, &ctx->gi_bcount, &ctx->svo_grid,
                          &ctx->svo_bricks};
    for (tgx_buffer* b : bufs) tgx_buffer_release(b);
    tgx_buffer* prev[] = {&ctx->svo_prev_keys, &ctx->svo_prev_off, &ctx->svo_prev_cand, &ctx->svo_old_bits,
                          &ctx->svo_old_mats, &ctx->svo_old_n, &ctx->svo_old_list_off, &ctx->svo_old_list,
                          &ctx->svo_arena};
    for (tgx_buffer* b : prev) tgx_buffer_release(b);
    ctx->svo_built = false;
    ctx->svo_prev_valid = false;
}

namespace {
/* Temporary device arrays of one build, carved from the context's build
 * arena (kept between builds, so a rebuild of a similar scene allocates
 * nothing). What does not fit is allocated on its own and freed when the
 * build ends, and the arena grows to the whole need for the next build. */
struct dbuf {
    void* p = nullptr;
    template <typename T> T* as() { return (T*)p; }
};
int dalloc(tgx_context* ctx, dbuf& b, size_t bytes, const char* what)
{
    bytes = (bytes + 255u) & ~(size_t)255u;
    if (bytes == 0) bytes = 256;
    if (ctx->svo_arena.ptr && ctx->svo_arena_used + bytes <= ctx->svo_arena.bytes) {
        b.p = (char*)ctx->svo_arena.ptr + ctx->svo_arena_used;
        ctx->svo_arena_used += bytes;
        return TGX_OK;
    }
    hipError_t e = hipMalloc(&b.p, bytes);
    if (e != hipSuccess) {
        b.p = nullptr;
        return tgx_fail(ctx, TGX_ERR_OUT_OF_MEMORY, "hipMalloc(%zu) for %s", bytes, what);
    }
    ctx->svo_arena_spill.push_back(b.p);
    ctx->svo_arena_spill_bytes += bytes;
    return TGX_OK;
}
/* Opens the arena for one build; on every exit frees the spills and
 * records the size the next build needs. */
struct arena_scope {
    tgx_context* ctx;
    explicit arena_scope(tgx_context* c) : ctx(c)
    {
        ctx->svo_arena_used = 0;
        ctx->svo_arena_spill_bytes = 0;
        if (ctx->svo_arena_want > ctx->svo_arena.bytes) {
            tgx_buffer_release(&ctx->svo_arena);
            if (tgx_buffer_reserve(ctx, &ctx->svo_arena, ctx->svo_arena_want, "svo build arena")) {
                tgx_buffer_release(&ctx->svo_arena);  /* the build spills instead */
                ctx->last_error.clear();
            }
        }
    }
    ~arena_scope()
    {
        if (!ctx->svo_arena_spill.empty()) {
            (void)hipStreamSynchronize(ctx->stream);
            for (void* p : ctx->svo_arena_spill) (void)hipFree(p);
            ctx->svo_arena_spill.clear();
            const size_t need = ctx->svo_arena_used + ctx->svo_arena_spill_bytes;
            ctx->svo_arena_want = need + need / 4u;
        }
    }
};
/* Pinned scratch of the SVO code: bytes [64, 192) of the context's pinned
 * page (bytes [0, 64) hold the visibility statistics readback). */
inline uint32_t* svo_pinned(tgx_context* ctx) { return (uint32_t*)((char*)ctx->host_pinned + 64); }
/* The arena as it was at construction, for a step that is run again with
 * larger arrays (what spilled stays until the build ends). */
struct arena_mark {
    tgx_context* ctx;
    size_t       used;
    explicit arena_mark(tgx_context* c) : ctx(c), used(c->svo_arena_used) {}
    void release() const { ctx->svo_arena_used = used; }
};
}  // namespace

extern "C" {

static int svo_build(tgx_context* ctx, const float mn[3], uint32_t depth, uint32_t flags, bool update);

int tgx_svo_build(tgx_context* ctx, const float mn[3], uint32_t depth, uint32_t flags)
{
    return svo_build(ctx, mn, depth, flags, false);
}

int tgx_svo_update(tgx_context* ctx, uint32_t* reused_leaves, uint32_t* voxelized_leaves)
{
    if (!ctx) return TGX_ERR_INVALID_ARG;
    ctx->last_error.clear();
    if (!ctx->svo_built) return tgx_fail(ctx, TGX_ERR_NOT_BUILT, "no SVO built: call tgx_svo_build first");
    const float mn[3] = {ctx->svo_info.min[0], ctx->svo_info.min[1], ctx->svo_info.min[2]};
    const int rc = svo_build(ctx, mn, ctx->svo_info.depth, ctx->svo_info.flags, ctx->dynamic && ctx->svo_prev_valid);
    if (!rc) {
        if (reused_leaves) *reused_leaves = ctx->svo_reused;
        if (voxelized_leaves) *voxelized_leaves = ctx->svo_info.n_leaves - ctx->svo_reused;
    }
    return rc;
}

static int svo_build(tgx_context* ctx, const float mn[3], uint32_t depth, uint32_t flags, bool update)
{
    if (ctx && ctx->n_graphs > 0)
        return tgx_fail(ctx, TGX_ERR_INVALID_ARG, "a frame graph uses the SVO: destroy it before rebuilding");
    if (!ctx || !mn) return TGX_ERR_INVALID_ARG;
    ctx->last_error.clear();
    if (!ctx->has_scene) return tgx_fail(ctx, TGX_ERR_NO_SCENE, "no scene uploaded");
    if (depth < TGX_SVO_MIN_DEPTH || depth > TGX_SVO_MAX_DEPTH)
        return tgx_fail(ctx, TGX_ERR_INVALID_ARG, "depth %u outside [%u, %u]", depth, TGX_SVO_MIN_DEPTH, TGX_SVO_MAX_DEPTH);
    for (int a = 0; a < 3; a++)
        if (!(mn[a] == floorf(mn[a])) || fabsf(mn[a]) + (float)(1u << depth) >= 16777216.0f)
            return tgx_fail(ctx, TGX_ERR_INVALID_ARG, "svo min must be integral and |min| + 2^depth < 2^24");
    TGX_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    ctx->svo_reused = 0;
    ctx->svo_built = false;
    /* The buffers stay allocated and are reused when large enough. An
     * update keeps the last build's leaves aside (double buffering). */
    if (update) {
        std::swap(ctx->svo_leaf_bits, ctx->svo_old_bits);
        std::swap(ctx->svo_leaf_mats, ctx->svo_old_mats);
        std::swap(ctx->svo_leaf_moff, ctx->svo_old_moff);
        std::swap(ctx->svo_leaf_wpre, ctx->svo_old_wpre);
        std::swap(ctx->svo_leaf_n, ctx->svo_old_n);
        std::swap(ctx->svo_list_off, ctx->svo_old_list_off);
        std::swap(ctx->svo_list, ctx->svo_old_list);
    } else {
        ctx->svo_prev_valid = false;
    }
    arena_scope arena(ctx);
    int rc;
    const uint32_t n_cptr = ctx->n_cluster_pointers;
    if (n_cptr == 0) return tgx_fail(ctx, TGX_ERR_NO_SCENE, "the scene has no clusters");
    const uint32_t leaf_level = depth - 5u;

    if ((rc = tgx_buffer_reserve(ctx, &ctx->svo_frames, sizeof(svo_frame) * (size_t)n_cptr, "svo frames"))) return rc;
    svo_frame* frames = (svo_frame*)ctx->svo_frames.ptr;
    dbuf nonempty;
    if ((rc = dalloc(ctx, nonempty, 4ull * n_cptr, "svo flags"))) return rc;
    {
        tgx_launch_scope s(ctx, "svo_frames_k");
        hipLaunchKernelGGL(svo_frames_k, dim3(blocks_for(n_cptr)), dim3(256), 0, ctx->stream,
                           (const tgx_object*)ctx->objects.ptr, (const uint32_t*)ctx->cluster_pointers.ptr,
                           (const uint32_t*)ctx->cluster_idx_to_object.ptr, (const uint32_t*)ctx->bits.ptr, n_cptr,
                           frames, nonempty.as<uint32_t>());
    }
    TGX_LAUNCH_CHECK(ctx, "svo_frames_k");

    /* Levels: the pairs of one level give the next one's, in two arrays that
     * take turns, and the nodes' bitmap. No count comes back in between: the
     * arrays hold 3 pairs per cluster pointer (rotated boxes on a noise scene
     * need 1.8) or what the last build needed, and a level that needs more is
     * found afterwards and the levels run again. */
    const uint32_t map_words = node_word(leaf_level + 1u);
    dbuf map;
    if ((rc = dalloc(ctx, map, 4ull * (SVO_CNT_N + 3ull * map_words), "svo node bitmap"))) return rc;
    uint32_t* cnt = map.as<uint32_t>();
    uint32_t* bits_of = cnt + SVO_CNT_N;
    uint32_t* pre = bits_of + map_words;
    uint32_t* popc = pre + map_words;
    uint32_t* h = svo_pinned(ctx);
    uint32_t leaf_cnt[2 * SVO_CNT_BASE];
    const uint32_t *leaf_coord = nullptr, *leaf_cptr = nullptr;
    uint64_t cap = 3ull * n_cptr + 4096ull;
    if (cap < ctx->svo_pairs_need) cap = ctx->svo_pairs_need + ctx->svo_pairs_need / 4u;
    for (;;) {
        if (cap > 0xF0000000ull) return tgx_fail(ctx, TGX_ERR_CAPACITY, "too many (node, cluster) pairs");
        const arena_mark mark(ctx);
        dbuf pairs[2];
        if ((rc = dalloc(ctx, pairs[0], 8ull * cap, "svo pairs")) || (rc = dalloc(ctx, pairs[1], 8ull * cap, "svo pairs")))
            return rc;
        hipLaunchKernelGGL(svo_levels_init_k, dim3(blocks_for(SVO_CNT_N + map_words)), dim3(256), 0, ctx->stream, cnt,
                           SVO_CNT_N + map_words);
        for (uint32_t l = 0; l < leaf_level; l++) {
            const uint32_t n_max = l ? (uint32_t)cap : n_cptr;
            const uint64_t blocks = ((uint64_t)n_max + EXPAND_PAIRS - 1u) / EXPAND_PAIRS;
            const uint32_t* in = pairs[l & 1u].as<uint32_t>();
            uint32_t* out = pairs[(l + 1u) & 1u].as<uint32_t>();
            tgx_launch_scope s(ctx, "svo_expand_k");
            hipLaunchKernelGGL(svo_expand_k, dim3((uint32_t)(blocks < EXPAND_BLOCKS ? blocks : EXPAND_BLOCKS)), dim3(EXPAND_BLOCK), 0,
                               ctx->stream, l ? in : (const uint32_t*)nullptr, in + cap, nonempty.as<uint32_t>(), cnt + l,
                               n_max, frames, mn[0], mn[1], mn[2], (float)(1u << (depth - l)), cnt + l + 1u, out,
                               out + cap, (uint32_t)cap, bits_of + node_word(l + 1u), level_words(l + 1u));
        }
        TGX_LAUNCH_CHECK(ctx, "svo_expand_k");
        const bool wide = map_words > SVO_ONE_BLOCK_MAX;
        if (wide) {
            hipLaunchKernelGGL(svo_popc_k, dim3(blocks_for(map_words)), dim3(256), 0, ctx->stream, bits_of, map_words, popc);
            if ((rc = tgx_prim_exclusive_scan_u32(ctx, popc, pre, map_words))) return rc;
        }
        hipLaunchKernelGGL(svo_number_k, dim3(1), dim3(1024), 0, ctx->stream, cnt, bits_of, map_words, leaf_level,
                           wide ? 1u : 0u, pre, h);
        TGX_LAUNCH_CHECK(ctx, "svo_number_k");
        TGX_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
        uint64_t need = 0;
        for (uint32_t l = 1; l <= leaf_level && need <= cap; l++) need = h[l] > need ? h[l] : need;
        ctx->svo_pairs_need = need;
        if (need <= cap) {
            memcpy(leaf_cnt, h, sizeof(leaf_cnt));
            leaf_coord = pairs[leaf_level & 1u].as<uint32_t>();
            leaf_cptr = leaf_coord + cap;
            break;
        }
        cap = need + need / 4u;
        mark.release();
    }
    const uint32_t n_leaf_pairs = leaf_cnt[leaf_level];
    const uint32_t leaf_base = leaf_cnt[SVO_CNT_BASE + leaf_level];
    const uint32_t total_nodes = leaf_cnt[SVO_CNT_BASE + leaf_level + 1u];
    const uint32_t n_leaves = total_nodes - leaf_base;

    if (total_nodes >= 0xFFFFFFu)
        return tgx_fail(ctx, TGX_ERR_CAPACITY, "the SVO has %u nodes; the limit is 2^24 - 2", total_nodes);
    if ((rc = tgx_buffer_reserve(ctx, &ctx->svo_nodes, sizeof(svo_gnode) * (size_t)total_nodes, "svo nodes"))) return rc;
    svo_gnode* nodes = (svo_gnode*)ctx->svo_nodes.ptr;
    dbuf leaf_keys, keys, keys2, pair_cptr, first;
    if ((rc = dalloc(ctx, leaf_keys, 4ull * n_leaves, "svo leaf keys")) ||
        (rc = dalloc(ctx, keys, 8ull * n_leaf_pairs, "svo pair keys")) ||
        (rc = dalloc(ctx, keys2, 8ull * n_leaf_pairs, "svo pair keys")) ||
        (rc = dalloc(ctx, pair_cptr, 4ull * n_leaf_pairs, "svo pairs")) ||
        (rc = dalloc(ctx, first, 4ull * (n_leaves + 1ull), "svo first pair")))
        return rc;
    {
        tgx_launch_scope s(ctx, "svo_nodes_k");
        hipLaunchKernelGGL(svo_nodes_k, dim3(blocks_for(32ull * map_words)), dim3(256), 0, ctx->stream, bits_of, pre,
                           map_words, leaf_level, leaf_base, nodes, leaf_keys.as<uint32_t>());
    }
    TGX_LAUNCH_CHECK(ctx, "svo_nodes_k");
    if (n_leaf_pairs) {
        uint32_t cptr_bits = 1u, leaf_bits_n = 1u;
        while (cptr_bits < 32u && (n_cptr - 1u) >> cptr_bits) cptr_bits++;
        while ((n_leaves - 1u) >> leaf_bits_n) leaf_bits_n++;
        hipLaunchKernelGGL(svo_pair_keys_k, dim3(blocks_for(n_leaf_pairs)), dim3(256), 0, ctx->stream, leaf_coord,
                           leaf_cptr, n_leaf_pairs, bits_of, pre, leaf_level, leaf_base, cptr_bits, keys.as<uint64_t>());
        TGX_LAUNCH_CHECK(ctx, "svo_pair_keys_k");
        if ((rc = tgx_prim_sort_keys_u64(ctx, keys.as<uint64_t>(), keys2.as<uint64_t>(), n_leaf_pairs,
                                         cptr_bits + leaf_bits_n)))
            return rc;
        hipLaunchKernelGGL(svo_pair_split_k, dim3(blocks_for(n_leaf_pairs)), dim3(256), 0, ctx->stream,
                           keys2.as<uint64_t>(), n_leaf_pairs, cptr_bits, pair_cptr.as<uint32_t>(),
                           first.as<uint32_t>());
        TGX_LAUNCH_CHECK(ctx, "svo_pair_split_k");
    }

    /* Leaves. */
    const size_t nl = n_leaves ? n_leaves : 1;
    if ((rc = tgx_buffer_reserve(ctx, &ctx->svo_leaf_bits, 4ull * TGX_SVO_BLOCK_WORDS * nl, "svo leaf bits")) ||
        (rc = tgx_buffer_reserve(ctx, &ctx->svo_leaf_moff, 4ull * (nl + 1), "svo material offsets")) ||
        (rc = tgx_buffer_reserve(ctx, &ctx->svo_leaf_wpre, 2ull * TGX_SVO_BLOCK_WORDS * nl, "svo material prefixes")) ||
        (rc = tgx_buffer_reserve(ctx, &ctx->svo_leaf_n, 4ull * nl, "svo leaf n")) ||
        (rc = tgx_buffer_reserve(ctx, &ctx->svo_list_off, 4ull * (nl + 1), "svo list offsets")))
        return rc;
    dbuf list_tmp, solid, many;
    if ((rc = dalloc(ctx, list_tmp, 4ull * (n_leaf_pairs ? n_leaf_pairs : 1), "svo list")) ||
        (rc = dalloc(ctx, solid, 4ull * nl, "svo solid counts")) || (rc = dalloc(ctx, many, 4ull * nl, "svo leaves")))
        return rc;
    dbuf reuse;
    if (update && n_leaves) {
        if ((rc = dalloc(ctx, reuse, 4ull * n_leaves, "svo reuse"))) return rc;
        hipLaunchKernelGGL(svo_match_k, dim3((n_leaves + 3u) / 4u), dim3(256), 0, ctx->stream,
                           leaf_keys.as<uint32_t>(), first.as<uint32_t>(), n_leaf_pairs,
                           n_leaves, pair_cptr.as<uint32_t>(), frames, (const uint8_t*)ctx->cl_dirty.ptr, (const uint32_t*)ctx->svo_prev_keys.ptr,
                           ctx->svo_prev_leaves, (const uint32_t*)ctx->svo_prev_off.ptr,
                           (const uint32_t*)ctx->svo_prev_cand.ptr, reuse.as<uint32_t>(), cnt + SVO_CNT_REUSED);
        TGX_LAUNCH_CHECK(ctx, "svo_match_k");
    }
    /* Leaf sampling in two passes: bits, lists and solid counts; then,
     * with the counts scanned into material offsets, the materials of the
     * solid voxels only. */
    const uint32_t quirk = (flags & TGX_SVO_FLAG_REFERENCE_CORNER_QUIRK) ? 1u : 0u;
    const uint32_t* rz = update ? reuse.as<uint32_t>() : nullptr;
    const uint32_t few = n_leaves >= LEAF_FEW_LEAVES ? LEAF_FEW : 0u;
    auto leaf_grid = [](uint32_t n, uint32_t per_leaf) {
        const uint32_t row = n < LEAF_ROW ? n : LEAF_ROW;
        return dim3(per_leaf * row, (n + row - 1u) / row);
    };
    static_assert((uint64_t)LEAF_PARTS * LEAF_ROW * LEAF_BLOCK < 1ull << 32, "lanes of a row");
    if (n_leaves) {
        tgx_launch_scope s(ctx, "svo_leaf_k");
        const bool sparse = n_leaf_pairs <= (uint64_t)LEAF_SPARSE * n_leaves;
        hipLaunchKernelGGL(sparse ? svo_leaf_k<LEAF_SPARSE_BLOCK> : svo_leaf_k<LEAF_BLOCK>, leaf_grid(n_leaves, 1u),
                           dim3(sparse ? LEAF_SPARSE_BLOCK : LEAF_BLOCK), 0, ctx->stream, nodes, leaf_base,
                           pair_cptr.as<uint32_t>(), first.as<uint32_t>(), n_leaf_pairs,
                           n_leaves, frames, (const uint32_t*)ctx->bits.ptr, mn[0], mn[1], mn[2], quirk,
                           (uint32_t*)ctx->svo_leaf_bits.ptr, solid.as<uint32_t>(), (uint16_t*)ctx->svo_leaf_wpre.ptr,
                           (uint32_t*)ctx->svo_leaf_n.ptr, list_tmp.as<uint32_t>(), nodes, rz,
                           (const uint32_t*)ctx->svo_old_bits.ptr, (const uint32_t*)ctx->svo_old_moff.ptr,
                           (const uint16_t*)ctx->svo_old_wpre.ptr, (const uint32_t*)ctx->svo_old_n.ptr,
                           (const uint32_t*)ctx->svo_old_list_off.ptr, (const uint32_t*)ctx->svo_old_list.ptr,
                           few, cnt + SVO_CNT_MANY, many.as<uint32_t>());
    }
    TGX_LAUNCH_CHECK(ctx, "svo_leaf_k");
    /* material offsets and list offsets, their totals read back together */
    uint32_t* moff = (uint32_t*)ctx->svo_leaf_moff.ptr;
    uint32_t* list_off = (uint32_t*)ctx->svo_list_off.ptr;
    const uint32_t* leaf_n = (const uint32_t*)ctx->svo_leaf_n.ptr;
    if (n_leaves <= SVO_ONE_BLOCK_MAX) {
        hipLaunchKernelGGL(svo_offsets_k, dim3(2), dim3(1024), 0, ctx->stream, solid.as<uint32_t>(), moff, leaf_n, list_off,
                           n_leaves, cnt, h);
    } else {
        if ((rc = tgx_prim_exclusive_scan_u32(ctx, solid.as<uint32_t>(), moff, n_leaves)) ||
            (rc = tgx_prim_exclusive_scan_u32(ctx, leaf_n, list_off, n_leaves)))
            return rc;
        hipLaunchKernelGGL(svo_wrap_k, dim3(blocks_for(n_leaves)), dim3(256), 0, ctx->stream, solid.as<uint32_t>(), moff,
                           n_leaves, cnt + SVO_CNT_WRAP);
        hipLaunchKernelGGL(svo_totals_k, dim3(1), dim3(64), 0, ctx->stream, solid.as<uint32_t>(), moff, leaf_n, list_off,
                           n_leaves, cnt, h);
    }
    TGX_LAUNCH_CHECK(ctx, "svo_offsets_k");
    TGX_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    if (h[4])
        return tgx_fail(ctx, TGX_ERR_CAPACITY, "the SVO's leaves hold 2^32 solid voxels or more; the limit is 2^32 - 1");
    const uint32_t n_solid = h[0], n_list = h[1];
    ctx->svo_reused = h[2];
    const uint32_t n_many = few ? h[3] : n_leaves;
    if ((rc = tgx_buffer_reserve(ctx, &ctx->svo_leaf_mats, 2ull * (n_solid ? n_solid : 1), "svo leaf materials")) ||
        (rc = tgx_buffer_reserve(ctx, &ctx->svo_list, 4ull * (n_list ? n_list : 1), "svo list")))
        return rc;
    ctx->svo_n_solid = n_solid;
    if (n_leaves) {
        tgx_launch_scope s(ctx, "svo_leaf_mats_k");
        auto mats = [&](auto kernel, dim3 blocks, uint32_t lanes, uint32_t limit) {
            hipLaunchKernelGGL(kernel, blocks, dim3(lanes), 0, ctx->stream, nodes, leaf_base,
                               pair_cptr.as<uint32_t>(), first.as<uint32_t>(), n_leaf_pairs, n_leaves, frames,
                               (const uint32_t*)ctx->bits.ptr, tgx_scene_materials(ctx), mn[0], mn[1], mn[2], quirk,
                               (const uint32_t*)ctx->svo_leaf_bits.ptr, (const uint16_t*)ctx->svo_leaf_wpre.ptr,
                               (const uint32_t*)ctx->svo_leaf_moff.ptr, (uint16_t*)ctx->svo_leaf_mats.ptr, rz,
                               (const uint32_t*)ctx->svo_old_moff.ptr, (const uint16_t*)ctx->svo_old_mats.ptr,
                               few ? many.as<uint32_t>() : (uint32_t*)nullptr, limit);
        };
        if (n_many < n_leaves) mats(svo_leaf_mats_few_k, leaf_grid(n_leaves, 1u), LEAF_FEW_BLOCK, few);
        if (n_many) mats(svo_leaf_mats_k, leaf_grid(n_many, LEAF_PARTS), LEAF_BLOCK, n_many);
    }
    TGX_LAUNCH_CHECK(ctx, "svo_leaf_mats_k");
    /* Lists; and the traversal layout: leaf brick masks and the leaf grid. */
    const uint32_t n_inner = leaf_base;
    if ((rc = tgx_buffer_reserve(ctx, &ctx->svo_grid, 4ull << (3u * leaf_level), "svo leaf grid")) ||
        (rc = tgx_buffer_reserve(ctx, &ctx->svo_bricks, 8ull * nl, "svo leaf bricks")))
        return rc;
    if (n_leaves)
        hipLaunchKernelGGL(svo_bricks_k, dim3((n_leaves + 3u) / 4u), dim3(256), 0, ctx->stream,
                           (const uint32_t*)ctx->svo_leaf_bits.ptr, n_leaves, (unsigned long long*)ctx->svo_bricks.ptr,
                           list_tmp.as<uint32_t>(), first.as<uint32_t>(), leaf_n, list_off, (uint32_t*)ctx->svo_list.ptr);
    TGX_LAUNCH_CHECK(ctx, "svo_bricks_k");
    hipLaunchKernelGGL(svo_grid_k, dim3(blocks_for(1ull << (3u * (leaf_level - 1u)))), dim3(256), 0, ctx->stream,
                       (const svo_gnode*)nodes, leaf_level, (const unsigned long long*)ctx->svo_bricks.ptr,
                       (uint32_t*)ctx->svo_grid.ptr);
    TGX_LAUNCH_CHECK(ctx, "svo_grid_k");
    if (ctx->dynamic) {
        /* what the next tgx_svo_update compares against */
        if ((rc = tgx_buffer_reserve(ctx, &ctx->svo_prev_keys, 4ull * nl, "svo previous keys")) ||
            (rc = tgx_buffer_reserve(ctx, &ctx->svo_prev_off, 4ull * (nl + 1), "svo previous offsets")) ||
            (rc = tgx_buffer_reserve(ctx, &ctx->svo_prev_cand, 4ull * (n_leaf_pairs ? n_leaf_pairs : 1), "svo previous candidates")))
            return rc;
        const uint64_t dirty_words = (ctx->n_clusters + 3ull) / 4ull;
        const uint64_t most = n_leaf_pairs > dirty_words ? n_leaf_pairs : dirty_words;
        hipLaunchKernelGGL(svo_keep_k, dim3(blocks_for(most + 1u)), dim3(256), 0, ctx->stream, leaf_keys.as<uint32_t>(),
                           first.as<uint32_t>(), n_leaves, pair_cptr.as<uint32_t>(), n_leaf_pairs, frames,
                           (uint32_t)dirty_words, (uint32_t*)ctx->svo_prev_keys.ptr, (uint32_t*)ctx->svo_prev_off.ptr,
                           (uint32_t*)ctx->svo_prev_cand.ptr, (uint32_t*)ctx->cl_dirty.ptr);
        TGX_LAUNCH_CHECK(ctx, "svo_keep_k");
        ctx->svo_prev_leaves = n_leaves;
    }
    TGX_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    ctx->svo_prev_valid = ctx->dynamic;
    ctx->svo_n_inner = n_inner;

    ctx->svo_info.min[0] = mn[0]; ctx->svo_info.min[1] = mn[1]; ctx->svo_info.min[2] = mn[2];
    ctx->svo_info.depth = depth;
    ctx->svo_info.n_nodes = total_nodes;
    ctx->svo_info.n_leaves = n_leaves;
    ctx->svo_info.n_list_entries = n_list;
    ctx->svo_info.flags = flags;
    ctx->svo_built = true;
    ctx->svo_stale = false;
    return TGX_OK;
}

int tgx_svo_device_bytes(tgx_context* ctx, uint64_t* bytes, uint64_t* solid_voxels)
{
    if (!ctx || !bytes) return TGX_ERR_INVALID_ARG;
    if (!ctx->svo_built) return tgx_fail(ctx, TGX_ERR_NOT_BUILT, "no SVO built");
    const tgx_svo_info& in = ctx->svo_info;
    const uint64_t nl = in.n_leaves;
    *bytes = (uint64_t)sizeof(svo_gnode) * in.n_nodes                  /* node records           */
             + (4ull * TGX_SVO_BLOCK_WORDS + 2ull * TGX_SVO_BLOCK_WORDS) * nl /* bits, word prefixes */
             + 4ull * (nl + 1) + 2ull * ctx->svo_n_solid               /* material offsets, pool */
             + 4ull * nl + 4ull * (nl + 1) + 4ull * in.n_list_entries  /* cluster lists          */
             + (4ull << (3u * (in.depth - 5u))) + 8ull * nl;           /* traversal layout       */
    if (solid_voxels) *solid_voxels = ctx->svo_n_solid;
    return TGX_OK;
}

int tgx_svo_get_info(tgx_context* ctx, tgx_svo_info* out)
{
    if (!ctx || !out) return TGX_ERR_INVALID_ARG;
    if (!ctx->svo_built) return tgx_fail(ctx, TGX_ERR_NOT_BUILT, "no SVO built");
    *out = ctx->svo_info;
    return TGX_OK;
}

}  /* extern "C" */

/* SVO files: "TGXSVO01", a header, the build's own node records, the leaf
 * counts, list offsets and lists, then per leaf its 1024 bit words and the
 * materials of its solid voxels only (in bit order), and an FNV-1a 64
 * checksum of everything before it. */
namespace {
struct svo_file_header {
    char         magic[8];
    uint32_t     version;
    uint32_t     n_inner;
    tgx_svo_info info;
    uint32_t     n_clusters;   /* of the scene the SVO was built from */
    uint32_t     n_luts;
    uint64_t     n_solid;      /* solid voxels over all leaves */
};
const char k_svo_magic[8] = {'T', 'G', 'X', 'S', 'V', 'O', '0', '1'};
constexpr uint32_t k_svo_chunk = 2048u;   /* leaves per staged chunk */

struct svo_stream {
    FILE*    f = nullptr;
    uint64_t h = 0xCBF29CE484222325ull;
    bool     bad = false;
    void hash(const void* p, size_t n)
    {
        const unsigned char* b = (const unsigned char*)p;
        for (size_t i = 0; i < n; i++) { h ^= b[i]; h *= 0x100000001B3ull; }
    }
    void put(const void* p, size_t n)
    {
        if (bad || (n && fwrite(p, 1, n, f) != n)) { bad = true; return; }
        hash(p, n);
    }
    void get(void* p, size_t n)
    {
        if (bad || (n && fread(p, 1, n, f) != n)) { bad = true; return; }
        hash(p, n);
    }
    ~svo_stream() { if (f) fclose(f); }
};

inline uint32_t popc32(uint32_t v) { return (uint32_t)__builtin_popcount(v); }

/* The invariants tgx_svo_build's layout guarantees and the traversal relies
 * on: every index a kernel follows stays inside its array. */
const char* check_svo_nodes(const std::vector<svo_gnode>& g, uint32_t n_inner, uint32_t depth)
{
    const uint32_t n = (uint32_t)g.size(), leaf_level = depth - 5u;
    if (n == 0 || n_inner == 0 || n_inner > n) return "node counts";
    if (g[0].parent != SVO_NONE || ((g[0].masks >> 16) & 0xFFu) != 0u || g[0].cx || g[0].cy || g[0].cz) return "root";
    uint64_t claimed = 0;   /* children named by some parent; each names its parent */
    for (uint32_t i = 0; i < n; i++) {
        const svo_gnode& a = g[i];
        const uint32_t lvl = (a.masks >> 16) & 0xFFu, valid = a.masks & 0xFFu, leafm = (a.masks >> 8) & 0xFFu;
        if (a.masks >> 24) return "node masks";
        if (i >= n_inner) {
            if (lvl != leaf_level || valid || leafm || a.first_child != SVO_NONE || a.leaf_idx != i - n_inner)
                return "leaf node";
            continue;
        }
        if (lvl >= leaf_level || a.leaf_idx != SVO_NONE) return "inner node";
        const uint32_t kids = popc32(valid);
        if (kids == 0) {
            if (a.first_child != SVO_NONE || leafm) return "childless node";
            continue;
        }
        claimed += kids;
        const bool at_leaves = lvl + 1u == leaf_level;
        if (leafm != (at_leaves ? valid : 0u)) return "leaf mask";
        const uint64_t f = a.first_child, e = f + kids;
        if (f <= i || e > (at_leaves ? n : n_inner) || (at_leaves && f < n_inner)) return "child range";
        uint32_t slot = 0;
        for (uint32_t rc = 0; rc < 8u; rc++) {
            if (!(valid & (1u << rc))) continue;
            const svo_gnode& c = g[f + slot++];
            if (c.parent != i || ((c.masks >> 16) & 0xFFu) != lvl + 1u || c.cx != 2u * a.cx + (rc & 1u) ||
                c.cy != 2u * a.cy + ((rc >> 1) & 1u) || c.cz != 2u * a.cz + (rc >> 2))
                return "child record";
        }
    }
    if (claimed != n - 1u) return "unreachable nodes";
    return nullptr;
}
}  // namespace

extern "C" {

int tgx_svo_save(tgx_context* ctx, const char* path)
{
    if (!ctx || !path) return TGX_ERR_INVALID_ARG;
    ctx->last_error.clear();
    /* the file records the scene's counts: a stale SVO would not match them */
    if (int rc0 = tgx_svo_check_current(ctx)) return rc0;
    TGX_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    TGX_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    const tgx_svo_info in = ctx->svo_info;
    const uint32_t nl = in.n_leaves;
    std::vector<svo_gnode> g(in.n_nodes);
    std::vector<uint32_t> leaf_n(nl), off(nl + 1u), list(in.n_list_entries);
    TGX_HIP_CHECK(ctx, hipMemcpy(g.data(), ctx->svo_nodes.ptr, sizeof(svo_gnode) * g.size(), hipMemcpyDeviceToHost));
    if (nl) TGX_HIP_CHECK(ctx, hipMemcpy(leaf_n.data(), ctx->svo_leaf_n.ptr, 4ull * nl, hipMemcpyDeviceToHost));
    TGX_HIP_CHECK(ctx, hipMemcpy(off.data(), ctx->svo_list_off.ptr, 4ull * (nl + 1u), hipMemcpyDeviceToHost));
    if (!list.empty())
        TGX_HIP_CHECK(ctx, hipMemcpy(list.data(), ctx->svo_list.ptr, 4ull * list.size(), hipMemcpyDeviceToHost));
    /* the leaves' materials are stored as in the file: solid voxels only,
     * in bit order, from the leaf's material offset */
    std::vector<uint32_t> moff(nl + 1u);
    TGX_HIP_CHECK(ctx, hipMemcpy(moff.data(), ctx->svo_leaf_moff.ptr, 4ull * (nl + 1u), hipMemcpyDeviceToHost));
    std::vector<uint32_t> bits((size_t)k_svo_chunk * TGX_SVO_BLOCK_WORDS);
    std::vector<uint16_t> mats;
    const uint64_t n_solid = moff[nl];
    svo_stream s;
    s.f = fopen(path, "wb");
    if (!s.f) return tgx_fail(ctx, TGX_ERR_IO, "cannot write %s", path);
    svo_file_header hd = {};
    memcpy(hd.magic, k_svo_magic, 8);
    hd.version = 1u;
    hd.n_inner = ctx->svo_n_inner;
    hd.info = in;
    hd.n_clusters = ctx->n_clusters;
    hd.n_luts = ctx->n_luts;
    hd.n_solid = n_solid;
    s.put(&hd, sizeof(hd));
    s.put(g.data(), sizeof(svo_gnode) * g.size());
    s.put(leaf_n.data(), 4ull * nl);
    s.put(off.data(), 4ull * (nl + 1u));
    s.put(list.data(), 4ull * list.size());
    for (uint32_t l0 = 0; l0 < nl && !s.bad; l0 += k_svo_chunk) {
        const uint32_t m = std::min(k_svo_chunk, nl - l0);
        TGX_HIP_CHECK(ctx, hipMemcpy(bits.data(), (const uint32_t*)ctx->svo_leaf_bits.ptr + (size_t)l0 * TGX_SVO_BLOCK_WORDS,
                                     4ull * TGX_SVO_BLOCK_WORDS * m, hipMemcpyDeviceToHost));
        mats.resize((size_t)moff[l0 + m] - moff[l0]);
        if (!mats.empty())
            TGX_HIP_CHECK(ctx, hipMemcpy(mats.data(), (const uint16_t*)ctx->svo_leaf_mats.ptr + moff[l0],
                                         2ull * mats.size(), hipMemcpyDeviceToHost));
        for (uint32_t k = 0; k < m; k++) {
            s.put(&bits[(size_t)k * TGX_SVO_BLOCK_WORDS], 4ull * TGX_SVO_BLOCK_WORDS);
            s.put(mats.data() + (moff[l0 + k] - moff[l0]), 2ull * (moff[l0 + k + 1] - moff[l0 + k]));
        }
    }
    const uint64_t h = s.h;
    s.put(&h, sizeof(h));
    if (s.bad) return tgx_fail(ctx, TGX_ERR_IO, "write error on %s", path);
    return TGX_OK;
}

int tgx_svo_load(tgx_context* ctx, const char* path)
{
    if (!ctx || !path) return TGX_ERR_INVALID_ARG;
    ctx->last_error.clear();
    if (ctx->n_graphs > 0)
        return tgx_fail(ctx, TGX_ERR_INVALID_ARG, "a frame graph uses the SVO: destroy it before loading");
    if (!ctx->has_scene) return tgx_fail(ctx, TGX_ERR_NO_SCENE, "load the SVO's scene first");
    svo_stream s;
    s.f = fopen(path, "rb");
    if (!s.f) return tgx_fail(ctx, TGX_ERR_IO, "cannot open %s", path);
    if (fseek(s.f, 0, SEEK_END) != 0) return tgx_fail(ctx, TGX_ERR_IO, "cannot seek in %s", path);
    const long fsize = ftell(s.f);
    rewind(s.f);
    svo_file_header hd;
    s.get(&hd, sizeof(hd));
    if (s.bad || memcmp(hd.magic, k_svo_magic, 8) != 0 || hd.version != 1u)
        return tgx_fail(ctx, TGX_ERR_INVALID_ARG, "%s is not an SVO file", path);
    const tgx_svo_info in = hd.info;
    /* the fixed-size parts must fit in the file before anything is allocated */
    const uint64_t fixed = sizeof(hd) + sizeof(svo_gnode) * (uint64_t)in.n_nodes + 4ull * (2ull * in.n_leaves + 1u) +
                           4ull * in.n_list_entries + 4ull * TGX_SVO_BLOCK_WORDS * in.n_leaves + 2ull * hd.n_solid + 8u;
    bool bad_min = false;
    for (int a = 0; a < 3; a++)
        bad_min |= !(in.min[a] == floorf(in.min[a])) ||
                   !(fabsf(in.min[a]) + (float)(1u << (in.depth & 15u)) < 16777216.0f);
    if (in.depth < TGX_SVO_MIN_DEPTH || in.depth > TGX_SVO_MAX_DEPTH || bad_min || in.n_nodes == 0 ||
        in.n_nodes >= 0xFFFFFFu || hd.n_inner > in.n_nodes || in.n_leaves != in.n_nodes - hd.n_inner ||
        hd.n_solid > (uint64_t)in.n_leaves * TGX_SVO_BLOCK_VOXELS || hd.n_solid > 0xFFFFFFFFull || fsize < 0 || fixed != (uint64_t)fsize)
        return tgx_fail(ctx, TGX_ERR_INVALID_ARG, "%s: inconsistent SVO header or file size", path);
    if (hd.n_clusters != ctx->n_clusters || hd.n_luts != ctx->n_luts)
        return tgx_fail(ctx, TGX_ERR_INVALID_ARG, "%s was built from a scene of %u clusters and %u LUTs, not %u and %u",
                        path, hd.n_clusters, hd.n_luts, ctx->n_clusters, ctx->n_luts);
    const uint32_t nl = in.n_leaves;
    std::vector<svo_gnode> g(in.n_nodes);
    std::vector<uint32_t> leaf_n(nl), off(nl + 1u), list(in.n_list_entries);
    s.get(g.data(), sizeof(svo_gnode) * g.size());
    s.get(leaf_n.data(), 4ull * nl);
    s.get(off.data(), 4ull * (nl + 1u));
    s.get(list.data(), 4ull * list.size());
    if (s.bad) return tgx_fail(ctx, TGX_ERR_INVALID_ARG, "%s is truncated", path);
    if (const char* why = check_svo_nodes(g, hd.n_inner, in.depth))
        return tgx_fail(ctx, TGX_ERR_INVALID_ARG, "%s: bad SVO nodes (%s)", path, why);
    if (off[0] != 0u || off[nl] != in.n_list_entries) return tgx_fail(ctx, TGX_ERR_INVALID_ARG, "%s: bad list offsets", path);
    for (uint32_t l = 0; l < nl; l++)
        if (off[l + 1] < off[l] || off[l + 1] - off[l] != leaf_n[l] ||
            g[hd.n_inner + l].leaf_n != leaf_n[l])
            return tgx_fail(ctx, TGX_ERR_INVALID_ARG, "%s: bad leaf lists", path);
    for (uint32_t c : list)
        if (c >= ctx->n_clusters) return tgx_fail(ctx, TGX_ERR_INVALID_ARG, "%s: cluster index out of range", path);
    for (const svo_gnode& a : g)
        if (a.leaf_n && a.leaf_idx == SVO_NONE) return tgx_fail(ctx, TGX_ERR_INVALID_ARG, "%s: bad node", path);

    /* Leaf data in two passes over the file: the first checks every leaf
     * and the checksum with nothing on the device touched, the second
     * uploads (and hashes again, against a file changed in between). */
    std::vector<uint32_t> bits((size_t)k_svo_chunk * TGX_SVO_BLOCK_WORDS), moff(nl + 1u);
    std::vector<uint16_t> mats, wpre((size_t)k_svo_chunk * TGX_SVO_BLOCK_WORDS);
    const long leaf_data_at = ftell(s.f);
    const uint64_t h_leaf = s.h;
    auto leaf_pass = [&](bool upload) -> int {
        uint64_t n_solid = 0;
        for (uint32_t l0 = 0; l0 < nl; l0 += k_svo_chunk) {
            const uint32_t m = std::min(k_svo_chunk, nl - l0);
            const uint64_t chunk_first = n_solid;
            mats.clear();
            for (uint32_t k = 0; k < m && !s.bad; k++) {
                uint32_t* b = &bits[(size_t)k * TGX_SVO_BLOCK_WORDS];
                s.get(b, 4ull * TGX_SVO_BLOCK_WORDS);
                uint32_t cnt = 0;
                for (uint32_t w = 0; w < TGX_SVO_BLOCK_WORDS; w++) {
                    wpre[(size_t)k * TGX_SVO_BLOCK_WORDS + w] = (uint16_t)cnt;
                    cnt += popc32(b[w]);
                }
                moff[l0 + k] = (uint32_t)n_solid;
                n_solid += cnt;
                if (s.bad || n_solid > hd.n_solid) { s.bad = true; break; }
                const size_t at = mats.size();
                mats.resize(at + cnt);
                s.get(mats.data() + at, 2ull * cnt);
                for (uint32_t j = 0; j < cnt && !s.bad; j++)
                    if (ctx->n_luts && (uint32_t)(mats[at + j] >> 8) >= ctx->n_luts) s.bad = true;
            }
            if (s.bad) return tgx_fail(ctx, TGX_ERR_INVALID_ARG, "%s: truncated or bad leaf data", path);
            if (!upload) continue;
            TGX_HIP_CHECK(ctx, hipMemcpy((uint32_t*)ctx->svo_leaf_bits.ptr + (size_t)l0 * TGX_SVO_BLOCK_WORDS,
                                         bits.data(), 4ull * TGX_SVO_BLOCK_WORDS * m, hipMemcpyHostToDevice));
            TGX_HIP_CHECK(ctx, hipMemcpy((uint16_t*)ctx->svo_leaf_wpre.ptr + (size_t)l0 * TGX_SVO_BLOCK_WORDS,
                                         wpre.data(), 2ull * TGX_SVO_BLOCK_WORDS * m, hipMemcpyHostToDevice));
            if (!mats.empty())
                TGX_HIP_CHECK(ctx, hipMemcpy((uint16_t*)ctx->svo_leaf_mats.ptr + chunk_first, mats.data(),
                                             2ull * mats.size(), hipMemcpyHostToDevice));
        }
        if (n_solid != hd.n_solid) return tgx_fail(ctx, TGX_ERR_INVALID_ARG, "%s: solid voxel count mismatch", path);
        moff[nl] = (uint32_t)n_solid;
        return TGX_OK;
    };
    int rc;
    if (leaf_data_at < 0) return tgx_fail(ctx, TGX_ERR_IO, "cannot tell the position in %s", path);
    if ((rc = leaf_pass(false))) return rc;
    const uint64_t h = s.h;
    uint64_t stored = 0;
    if (fread(&stored, sizeof(stored), 1, s.f) != 1 || stored != h)
        return tgx_fail(ctx, TGX_ERR_INVALID_ARG, "%s: checksum mismatch", path);

    TGX_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    TGX_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    ctx->svo_built = false;
    ctx->svo_prev_valid = false;
    ctx->svo_reused = 0;
    const size_t nlr = nl ? nl : 1;
    if ((rc = tgx_buffer_reserve(ctx, &ctx->svo_nodes, sizeof(svo_gnode) * g.size(), "svo nodes")) ||
        (rc = tgx_buffer_reserve(ctx, &ctx->svo_leaf_bits, 4ull * TGX_SVO_BLOCK_WORDS * nlr, "svo leaf bits")) ||
        (rc = tgx_buffer_reserve(ctx, &ctx->svo_leaf_mats, 2ull * (hd.n_solid ? hd.n_solid : 1), "svo leaf materials")) ||
        (rc = tgx_buffer_reserve(ctx, &ctx->svo_leaf_moff, 4ull * (nlr + 1), "svo material offsets")) ||
        (rc = tgx_buffer_reserve(ctx, &ctx->svo_leaf_wpre, 2ull * TGX_SVO_BLOCK_WORDS * nlr, "svo material prefixes")) ||
        (rc = tgx_buffer_reserve(ctx, &ctx->svo_leaf_n, 4ull * nlr, "svo leaf n")) ||
        (rc = tgx_buffer_reserve(ctx, &ctx->svo_list_off, 4ull * (nlr + 1), "svo list offsets")) ||
        (rc = tgx_buffer_reserve(ctx, &ctx->svo_list, 4ull * (list.empty() ? 1 : list.size()), "svo list")) ||
        (rc = tgx_buffer_reserve(ctx, &ctx->svo_grid, 4ull << (3u * (in.depth - 5u)), "svo leaf grid")) ||
        (rc = tgx_buffer_reserve(ctx, &ctx->svo_bricks, 8ull * nlr, "svo leaf bricks")))
        return rc;
    if (fseek(s.f, leaf_data_at, SEEK_SET) != 0) return tgx_fail(ctx, TGX_ERR_IO, "cannot seek in %s", path);
    s.h = h_leaf;
    if ((rc = leaf_pass(true))) return rc;
    if (s.h != h) return tgx_fail(ctx, TGX_ERR_INVALID_ARG, "%s changed while loading", path);
    TGX_HIP_CHECK(ctx, hipMemcpy(ctx->svo_leaf_moff.ptr, moff.data(), 4ull * (nl + 1u), hipMemcpyHostToDevice));
    ctx->svo_n_solid = hd.n_solid;
    TGX_HIP_CHECK(ctx, hipMemcpy(ctx->svo_nodes.ptr, g.data(), sizeof(svo_gnode) * g.size(), hipMemcpyHostToDevice));
    if (nl) TGX_HIP_CHECK(ctx, hipMemcpy(ctx->svo_leaf_n.ptr, leaf_n.data(), 4ull * nl, hipMemcpyHostToDevice));
    TGX_HIP_CHECK(ctx, hipMemcpy(ctx->svo_list_off.ptr, off.data(), 4ull * (nl + 1u), hipMemcpyHostToDevice));
    if (!list.empty())
        TGX_HIP_CHECK(ctx, hipMemcpy(ctx->svo_list.ptr, list.data(), 4ull * list.size(), hipMemcpyHostToDevice));
    if (nl)
        hipLaunchKernelGGL(svo_bricks_k, dim3((nl + 3u) / 4u), dim3(256), 0, ctx->stream,
                           (const uint32_t*)ctx->svo_leaf_bits.ptr, nl, (unsigned long long*)ctx->svo_bricks.ptr,
                           (const uint32_t*)nullptr, (const uint32_t*)nullptr, (const uint32_t*)nullptr,
                           (const uint32_t*)nullptr, (uint32_t*)nullptr);
    TGX_LAUNCH_CHECK(ctx, "svo_bricks_k");
    hipLaunchKernelGGL(svo_grid_k, dim3(blocks_for(1ull << (3u * (in.depth - 6u)))), dim3(256), 0, ctx->stream,
                       (const svo_gnode*)ctx->svo_nodes.ptr, in.depth - 5u,
                       (const unsigned long long*)ctx->svo_bricks.ptr, (uint32_t*)ctx->svo_grid.ptr);
    TGX_LAUNCH_CHECK(ctx, "svo_grid_k");
    TGX_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    ctx->svo_info = in;
    ctx->svo_n_inner = hd.n_inner;
    ctx->svo_built = true;
    ctx->svo_stale = false;
    return TGX_OK;
}

int tgx_svo_export(tgx_context* ctx, tgx_svo_node* nodes_out, uint32_t* leaf_bits, uint16_t* leaf_materials,
                   uint32_t* leaf_n, uint32_t* list_offsets, uint32_t* list)
{
    if (!ctx) return TGX_ERR_INVALID_ARG;
    if (!ctx->svo_built) return tgx_fail(ctx, TGX_ERR_NOT_BUILT, "no SVO built");
    const tgx_svo_info& in = ctx->svo_info;
    TGX_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    if (nodes_out) {
        std::vector<svo_gnode> g(in.n_nodes);
        TGX_HIP_CHECK(ctx, hipMemcpy(g.data(), ctx->svo_nodes.ptr, sizeof(svo_gnode) * in.n_nodes, hipMemcpyDeviceToHost));
        for (uint32_t i = 0; i < in.n_nodes; i++) {
            tgx_svo_node& o = nodes_out[i];
            o.level = (g[i].masks >> 16) & 0xFFu;
            o.coord[0] = g[i].cx; o.coord[1] = g[i].cy; o.coord[2] = g[i].cz;
            o.valid_mask = g[i].masks & 0xFFu;
            o.leaf_mask = (g[i].masks >> 8) & 0xFFu;
            o.first_child = g[i].first_child;
            o.leaf_idx = g[i].leaf_idx;
        }
    }
    if (leaf_bits && in.n_leaves)
        TGX_HIP_CHECK(ctx, hipMemcpy(leaf_bits, ctx->svo_leaf_bits.ptr, 4ull * TGX_SVO_BLOCK_WORDS * in.n_leaves, hipMemcpyDeviceToHost));
    if (leaf_materials && in.n_leaves) {
        /* the dense canonical grid from the solid voxels' materials */
        const uint32_t nl = in.n_leaves;
        std::vector<uint32_t> moff(nl + 1u), bw((size_t)k_svo_chunk * TGX_SVO_BLOCK_WORDS);
        std::vector<uint16_t> pm;
        TGX_HIP_CHECK(ctx, hipMemcpy(moff.data(), ctx->svo_leaf_moff.ptr, 4ull * (nl + 1u), hipMemcpyDeviceToHost));
        for (uint32_t l0 = 0; l0 < nl; l0 += k_svo_chunk) {
            const uint32_t m = std::min(k_svo_chunk, nl - l0);
            TGX_HIP_CHECK(ctx, hipMemcpy(bw.data(), (const uint32_t*)ctx->svo_leaf_bits.ptr + (size_t)l0 * TGX_SVO_BLOCK_WORDS,
                                         4ull * TGX_SVO_BLOCK_WORDS * m, hipMemcpyDeviceToHost));
            pm.resize((size_t)moff[l0 + m] - moff[l0]);
            if (!pm.empty())
                TGX_HIP_CHECK(ctx, hipMemcpy(pm.data(), (const uint16_t*)ctx->svo_leaf_mats.ptr + moff[l0],
                                             2ull * pm.size(), hipMemcpyDeviceToHost));
            uint16_t* out = leaf_materials + (size_t)l0 * TGX_SVO_BLOCK_VOXELS;
            memset(out, 0, 2ull * TGX_SVO_BLOCK_VOXELS * m);
            size_t j = 0;
            for (size_t w = 0; w < (size_t)m * TGX_SVO_BLOCK_WORDS; w++)
                for (uint32_t word = bw[w]; word; word &= word - 1u)
                    out[32u * w + (uint32_t)__builtin_ctz(word)] = pm[j++];
        }
    }
    if (leaf_n && in.n_leaves)
        TGX_HIP_CHECK(ctx, hipMemcpy(leaf_n, ctx->svo_leaf_n.ptr, 4ull * in.n_leaves, hipMemcpyDeviceToHost));
    if (list_offsets)
        TGX_HIP_CHECK(ctx, hipMemcpy(list_offsets, ctx->svo_list_off.ptr, 4ull * (in.n_leaves + 1), hipMemcpyDeviceToHost));
    if (list && in.n_list_entries)
        TGX_HIP_CHECK(ctx, hipMemcpy(list, ctx->svo_list.ptr, 4ull * in.n_list_entries, hipMemcpyDeviceToHost));
    return TGX_OK;
}

} /* extern "C" */
