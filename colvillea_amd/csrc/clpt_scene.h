/*
 * clpt_scene.h -- device-resident scene and wavefront layout (host/device
 * PODs).  Everything lives in HBM as flat arrays addressed by 32-bit
 * indices; all per-ray state is structure-of-arrays in float4 planes so a
 * wave64 reads and writes whole 1 KiB lines.
 */
#ifndef CLPT_SCENE_H
#define CLPT_SCENE_H

#include <hip/hip_runtime.h>
#include <stdint.h>

/* ---- BVH4 node as the builder makes it: float child boxes, stored per axis
 * (SoA inside the node).  Traversal reads its packed form, Node4P. ---- */
struct alignas(128) Node4
{
    float    lox[4], hix[4];
    float    loy[4], hiy[4];
    float    loz[4], hiz[4];
    uint32_t child[4];
    uint32_t pad[4];
};
static_assert(sizeof(Node4) == 128, "Node4 is two 64-byte halves");

/* ---- The BVH4 node as traversal reads it: 80 bytes, five 16-byte loads
 * instead of the float boxes' seven, packed on the device from Node4
 * (pack_node4).  A child's planes on axis a are p[a] + q s, q a half float
 * rounded outward after the box was widened by 2^-20 of the node's extent,
 * which covers the rounding of the slab test's arithmetic on them: a packed
 * box culls nothing that the float box keeps, so hits are the same bits
 * (checked for directions of length 1e-20 to 1e20 and extents of 1e-30 to
 * 1e37; boxes of nodes of 2^60 and more take every ray).
 * Empty slots hold an inverted infinite box. ---- */
struct alignas(16) Node4P
{
    uint16_t pl[3][2][4]; /* [axis][lo, hi][child], half bits */
    float    p[3], s;
    uint32_t child[4];
};
static_assert(sizeof(Node4P) == 80, "Node4P is five 16-byte words");

/* ---- BVH8 node: 96 bytes, read as 6 dwordx4.  Child boxes are stored
 * relative to the node's lower corner p, quantised to bytes per axis with a
 * power-of-two scale 2^(e - 127): child c spans
 *   [p + qlo[a][c] * 2^(e_a - 127), p + qhi[a][c] * 2^(e_a - 127)]
 * on axis a, evaluated in float32 exactly as written (a product of a byte
 * and a power of two is exact; the sum rounds once).  The builder picks the
 * bytes so that the decoded box contains the child's true box.  Empty slots
 * have child = CLPT_CHILD_EMPTY. ---- */
struct alignas(16) Node8
{
    float    p[3];
    uint8_t  e[3];
    uint8_t  pad;
    uint8_t  qlo[3][8];
    uint8_t  qhi[3][8];
    uint32_t child[8];
};
static_assert(sizeof(Node8) == 96, "Node8 is six 16-byte words");

/* Child reference encoding. */
#define CLPT_CHILD_EMPTY 0xffffffffu
#define CLPT_LEAF_BIT 0x80000000u
#define CLPT_INST_BIT 0x40000000u
/* triangle leaf: LEAF | (count-1) << 27 | first triangle (27 bits) */
#define CLPT_TRI_LEAF(first, count) (CLPT_LEAF_BIT | ((uint32_t)((count)-1) << 27) | (uint32_t)(first))
#define CLPT_INST_LEAF(idx) (CLPT_LEAF_BIT | CLPT_INST_BIT | (uint32_t)(idx))
/* Mesh-tree leaves hold at most 2 triangles: the closest-hit kernel tests
 * one triangle per step beside its node visits, and 2 measured slightly
 * faster than 4 (1 costs 4% more node visits). */
#define CLPT_MAX_LEAF_TRIS 2u

/* Traversal stack: CLPT_LDS_STACK entries per lane in LDS, the rest (up to
 * CLPT_STACK_TOTAL) in a global overflow area of (ref, t) pairs. */
#define CLPT_LDS_STACK 12
#define CLPT_STACK_TOTAL 128
#define CLPT_GSTACK_ENTRIES (CLPT_STACK_TOTAL - CLPT_LDS_STACK)
#define CLPT_MAX_TRIS (1u << 27)
#define CLPT_MAX_INSTANCES 0x3ffffff0u

/* Triangle in leaf order: v0.xyz + original primitive index (bits), v1, v2. */
struct TriRec
{
    float4 v0p;
    float4 v1;
    float4 v2;
};

struct alignas(16) InstanceRec
{
    float    xf[12];  /* object -> world */
    float    inv[12]; /* world -> object */
    uint32_t blas_root;
    uint32_t mesh;
    uint32_t material;
    uint32_t entity;
    uint32_t shade_off;  /* the mesh's first ShadeRec */
    uint32_t mesh_flags; /* MESH_HAS_* */
    uint32_t mtl_type;   /* the material's type */
    uint32_t pad;
};
static_assert(sizeof(InstanceRec) == 128, "InstanceRec is one 128-byte line");

/* What shading reads of a hit triangle, in original triangle order: vertex
 * positions, normals and uvs (zeros where the mesh has none) in one 128-byte
 * line, built on the device from the indexed arrays.  Through the arrays a
 * hit read its indices and then six places of vertices. */
struct alignas(128) ShadeRec
{
    float p[3][3];
    float n[3][3];
    float uv[3][2];
    float pad[8];
};
static_assert(sizeof(ShadeRec) == 128, "ShadeRec is one 128-byte line");

enum : uint32_t
{
    MESH_HAS_NORMALS  = 1u,
    MESH_HAS_TANGENTS = 2u,
    MESH_HAS_UVS      = 4u
};

struct MeshRec
{
    uint32_t idx_off; /* first index (x3) in the global index array */
    uint32_t vtx_off; /* first vertex in the global vertex arrays */
    uint32_t ntris;
    uint32_t flags;
};

/* Material: type, reflectance, GGX alpha = max(roughness^2, 1e-4), eta, k,
 * ior, and texture ids + 1 (0 = none) for the reflectance, the roughness
 * and the normal map. */
struct alignas(16) MaterialRec
{
    uint32_t type;
    float    r[3];
    float    alpha;
    float    eta[3];
    float    k[3];
    float    ior;
    uint32_t tex_r, tex_rough, tex_n, pad;
};
static_assert(sizeof(MaterialRec) == 64, "MaterialRec is four 16-byte words");

/* An RGBA32F texture: texels row-major, row 0 at v = 0. */
struct alignas(16) TexRec
{
    const float4* data;
    uint32_t      w, h;
};

struct alignas(16) EmitterRec
{
    uint32_t type;
    float    intensity[3];
    float    dir[3];
    float    tan_r; /* tan(angular radius) rounded once on the host */
};

/* Buckets of the HDRI CDF search cut points (SceneView::cutv, cutcond). */
#define CLPT_CUTS 1024u

/* Everything a kernel needs to find the scene; passed by value. */
struct SceneView
{
    const void*        nodes; /* Node4P or Node8 array (the tree width is a kernel template argument) */
    const TriRec*      tris;
    const InstanceRec* inst;
    const MeshRec*     meshes;
    const ShadeRec*    shade; /* per triangle of every mesh */
    const float*       tan;   /* xyz per vertex, read through idx */
    const uint32_t*    idx;
    const MaterialRec* mtl;
    const TexRec*      tex; /* material textures by id */
    uint32_t           ntex;
    const EmitterRec*  emitters;
    uint32_t           nemitters;
    int32_t            dome_index;
    const float4*      dome_tex; /* rgb and, in w, the texel's value of the sampling function (pcond) */
    uint32_t           dome_w, dome_h;
    const float*       cdfcond;
    const float*       pv;
    const float*       cdfv;
    const uint32_t*    cutv;    /* CLPT_CUTS + 1 search cut points of cdfv */
    const uint32_t*    cutcond; /* CLPT_CUTS + 1 per row of cdfcond */
    uint32_t           tlas_root;
    uint32_t           world_inst; /* the instance whose mesh subtrees the top tree holds (its
                                      transform is the identity), or 0xffffffff */
    uint32_t           ninst;
    uint32_t           bvh_width; /* 4 (Node4P) or 8 (Node8) */
    uint32_t           node_bytes; /* size of the node array (below 4 GiB) */
    uint32_t           stack_need; /* most stack entries a ray can hold (at most CLPT_STACK_TOTAL) */
};

/* One camera view: film size, path depth, RNG view lane, the view's offset
 * in the float64 film, and the camera basis (core::Camera, camera.h:8-27). */
struct alignas(16) ViewRec
{
    uint32_t width, height, npix, max_depth;
    uint32_t rr_depth, lane, film_offset, pad;
    float    pos[4], d00[4], ddu[4], ddv[4];
};

/* A batch is a list of (view, first path, first sample, samples) entries;
 * path p of the batch belongs to the last entry with path_begin <= p.  Its
 * local index l = p - path_begin runs over groups of `group` pixels of the
 * view (BatchTable; in tile order), within a group over the entry's samples
 * and within a sample over the group's pixels, so that all samples of a
 * group are traced together and find its triangles and texels in the caches.
 * The batch to run is read from *cursor, which k_batch_end advances, so a
 * captured batch graph replays unchanged. */
struct BatchEntry
{
    uint32_t view, path_begin, sample_base, nsamples;
};

struct BatchRec
{
    uint32_t entry_off, nentries, npaths, pad;
};

/* Shading waits for the texels, vertices and HDRI entries it gathers, and a
 * group's samples gather the same ones.  1024 pixels (four 16 x 16 tiles, one
 * window of the queues) against whole samples of the film: C1 frame at 1080p
 * and 64 spp 77.0 -> 75.7 ms (shading 14.4 -> 13.5), 16 spp at 512 x 512
 * 2.28 -> 2.21, 48 views 63.9 -> 62.9; 256 and 8192 pixels are within 1%. */
#define CLPT_PIXEL_GROUP 1024u
struct BatchTable
{
    const ViewRec*    views;
    const BatchRec*   batches;
    const BatchEntry* entries;
    uint32_t*         cursor;
    uint32_t          group; /* pixels whose samples are traced together */
    uint32_t          tile; /* 1: paths of a sample in pixel rows; T > 1: in T x T tiles */
};

/* A ray queue: 3 float4 planes of CLPT_SEGS x seg_cap slots. */
struct RayQueue
{
    float4*   o;  /* origin.xyz, w unused (read by traversal only) */
    float4*   d;  /* direction.xyz, path id (bits) */
    float4*   T;  /* throughput.xyz, previous BSDF pdf (read by shading only; not
                     written for camera paths, whose throughput is 1 and pdf 0) */
    uint32_t  seg_cap; /* slots of a segment; segment s starts at slot s * seg_cap */
};

/* Closest hit of each ray: b1, b2, instance (bits; CLPT_NO_HIT for a miss),
 * original primitive index (bits).  Shading needs no hit distance. */
#define CLPT_NO_HIT 0xffffffffu
struct HitBuf
{
    float4* h;
};

struct ShadowQueue
{
    float4*   o; /* origin.xyz, Lo.r */
    float4*   d; /* direction.xyz, Lo.g */
    float2*   x; /* Lo.b, pixel (bits) */
    uint32_t* tag; /* training record of the shadow ray (guided shading only; else NULL) */
};

/* ---- learned directional proposal ---- */

/* A training sample: query (9), sampled direction (3), weight. */
struct GuideSample
{
    float4 a; /* q0..q3 */
    float4 b; /* q4..q7 */
    float4 c; /* q8, wi.xyz */
    float4 d; /* weight, unused */
};

/* Device state of online training. */
struct GuideCounters
{
    uint32_t           count;   /* samples gathered since the last step (may exceed the buffer) */
    uint32_t           trained; /* samples in the last step */
    uint32_t           steps;   /* Adam steps taken */
    float              wsum;    /* weight sum of the last step */
    float              loss;    /* weighted negative log-likelihood of the last step (per unit weight) */
    uint32_t           pad;
    unsigned long long samples_total;
    uint32_t           amax[4]; /* max hidden activation of each layer in the last step (float bits) */
};

/* What the guided shading kernels need.  Training records, per vertex depth
 * j and recorded path (slot), at rec = j * nslots + slot: V is 4 planes of
 * float4, plane k at k * (CLPT_MAXD + 1) * nslots (query q0..q8, the
 * sampled direction, then p_mix and R = f cos / T_next per channel; p_mix =
 * 0 marks no record), and E[rec] the contribution (rgb) that arrived at
 * depth j (escape of ray j or the shadow ray of vertex j). */
struct GuideView
{
    const __bf16*  img;  /* packed bf16 weights */
    const uint8_t* img8; /* packed e4m3 weights (FP8 inference), else NULL */
    const float*   scl;  /* FP8 scales (10 floats) */
    float         lo[3], inv_ext[3];
    float         c_bsdf; /* probability of BSDF sampling at guided vertices */
    uint32_t      nslots; /* recorded paths per batch (0 = no recording) */
    float4*       V;
    float4*       E;
    uint32_t*     gcount; /* gather scratch: samples per recorded path */
    uint32_t*     gblock; /* gather scratch: per-256-path block counts, then offsets */
};

#define CLPT_MAXD 32
/* The ray and shadow queues are CLPT_SEGS segments of seg_cap slots each,
 * with a count of their own: shading block b reads segment b % CLPT_SEGS and
 * appends to the same segment of the output queues, so a segment never
 * receives more rays than it held (camera paths are dealt to the segments in
 * windows of CLPT_SEG_WIN).  Slots are reserved by one atomic per wave, and
 * atomics of all XCDs on one word complete one per 12.7 ns: with a single
 * count they were the whole shading time, 1.65 ms per 8.3 M rays of a closed
 * room.  With a count per XCD, in a line of its own (blocks are dealt to the
 * 8 XCDs round robin, so a segment stays with one XCD), shading of a 1080p
 * 64-spp frame takes 16.0 ms instead of 24.9 and of the room (4 spp) 7.3
 * instead of 14.5; 16, 32 and 64 segments measure no faster than 8. */
#define CLPT_SEGS 8u
#define CLPT_SEG_WIN 1024u

/* Queue counts of one segment in one batch.  The rays of depth d + 1 and the
 * shadow rays of depth d are interleaved (rs[2 d] = shadow rays of depth d,
 * rs[2 d + 1] = rays of depth d + 1), so that shading reserves both of its
 * output queues with one 64-bit atomic on &rs[2 d]. */
struct alignas(256) SegCounters
{
    uint32_t rs[2 * (CLPT_MAXD + 2)];
};
struct BatchCounters
{
    SegCounters seg[CLPT_SEGS];
};

/* The segment of window w of a batch's camera paths: each group of CLPT_SEGS
 * consecutive windows goes to all segments once, in an order rotated by a
 * hash of the group (unrotated, a film whose rows hold a multiple of
 * CLPT_SEGS windows gives each segment one band of columns, which made a
 * 512x512 16-spp frame 3.3 instead of 2.8 ms). */
__host__ __device__ inline uint32_t seg_of_window(uint32_t w)
{
    return (w + ((w / CLPT_SEGS * 0x9E3779B1u) >> 24)) % CLPT_SEGS;
}

/* slots of a segment for a batch of at most `paths` paths */
__host__ __device__ inline uint32_t seg_slots(uint64_t paths)
{
    const uint64_t w = (paths + CLPT_SEG_WIN - 1u) / CLPT_SEG_WIN;
    return (uint32_t)((w + CLPT_SEGS - 1u) / CLPT_SEGS) * CLPT_SEG_WIN;
}

/* rays of depth d >= 1, shadow rays of depth d in segment s */
__host__ __device__ inline uint32_t* bc_rays(BatchCounters* bc, uint32_t s, uint32_t d) { return &bc->seg[s].rs[2 * d - 1]; }
__host__ __device__ inline uint32_t* bc_shadow(BatchCounters* bc, uint32_t s, uint32_t d) { return &bc->seg[s].rs[2 * d]; }
__host__ __device__ inline unsigned long long* bc_push(BatchCounters* bc, uint32_t s, uint32_t d)
{
    return reinterpret_cast<unsigned long long*>(&bc->seg[s].rs[2 * d]);
}

/* A render's traversal counts, kept per wave of the persistent traversal
 * grids: row r, wave w at c[r * stride + w].  Each wave adds to its own words
 * with plain loads and stores (launches on the stream do not overlap), and
 * the rows are summed when the counters are read.  One atomic per wave and
 * counter on shared words instead cost 13.5 ns each (words shared by the
 * eight XCDs move between their L2s): 137 us at the end of a closest-hit
 * launch of 50 rays and 168 us of an any-hit launch of 47. */
struct WaveCounts
{
    unsigned long long* c;
    uint32_t            stride;
};
enum : uint32_t
{
    CLPT_WC_TRACE_NODES  = 0u,
    CLPT_WC_TRACE_TRIS   = 1u,
    CLPT_WC_SHADOW_NODES = 2u,
    CLPT_WC_SHADOW_TRIS  = 3u
};
/* rows of depth d in 1..CLPT_MAXD, and the rows a render to depth d uses */
__host__ __device__ inline uint32_t wc_hits(uint32_t d) { return 2u + 2u * d; }
__host__ __device__ inline uint32_t wc_visible(uint32_t d) { return 3u + 2u * d; }
__host__ __device__ inline uint32_t wc_rows(uint32_t d) { return 4u + 2u * d; }

struct TotalCounters
{
    unsigned long long rays[CLPT_MAXD + 2];
    unsigned long long hits[CLPT_MAXD + 2];
    unsigned long long shadow[CLPT_MAXD + 2];
    unsigned long long visible[CLPT_MAXD + 2];
    unsigned long long trace_nodes, trace_tris, shadow_nodes, shadow_tris;
};

#endif
