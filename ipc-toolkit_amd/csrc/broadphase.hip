// Broad phase on the GPU: conservative boxes, 63-bit Morton codes, LBVH
// (Karras 2012 hierarchy, boxes refit in three steps) and candidate traversal.
//
// Boxes follow aabb.cpp:35-126 (nextafter(p -/+ r) outward in FP64, unions
// for edges and faces) and lbvh.cpp:29-41 (FP32 with one more outward ulp).
// Morton codes follow lbvh.cpp:148-169 (FP64 box centre mapped by the mesh
// box of the vertex boxes, morton.hpp:53-63) and are sorted stably, so a
// pair's orientation (query = lower sorted position, lbvh.cpp:413-424) is
// the one the CPU restatement produces.  The candidate set itself is every
// leaf pair whose FP32 boxes overlap and passes the filters, independent of
// the tree shape.
//
// Tree layout: internal node j (splitting sorted keys j | j+1) stores both
// child boxes, child links and the children's rightmost leaf positions in
// one 64-byte line, so a traversal step is one line load.
#include "context.hpp"
#include "shard.hpp"
#include "geometry.hpp"
#include "sort.hpp"

#include <utility>

namespace ipcg {

namespace {

constexpr int BP_BLOCK = 256;
constexpr int TR_BLOCK = 128;
constexpr int TR_STACK = 64;  // lbvh.cpp:378 MAX_STACK_SIZE
constexpr int TR_LSTACK = 16; // entries per lane kept in LDS; the rest in HBM
constexpr int64_t TR_FEW = 1 << 18, TR_FEWER = 1 << 16; // queries: see wave_queries
constexpr int TR_SHARE = 2;   // steps between two chances of idle lanes to take over subtrees
constexpr int TR_IDLE = 4;    // idle lanes that make it worth the exchange
constexpr int TR_QUEUE = 256; // overlapping leaves that a wave holds before it settles them

// AABB::from_point (+ swept union), aabb.cpp:21-55
__device__ __forceinline__ void vbox(const double* X0, const double* X1, int nV, int i, double r,
                                     double* lo, double* hi)
{
    const d3 p = ldx(X0, nV, i);
    lo[0] = nextafter(p.x - r, -INFINITY);
    lo[1] = nextafter(p.y - r, -INFINITY);
    lo[2] = nextafter(p.z - r, -INFINITY);
    hi[0] = nextafter(p.x + r, INFINITY);
    hi[1] = nextafter(p.y + r, INFINITY);
    hi[2] = nextafter(p.z + r, INFINITY);
    if (X1) {
        const d3 q = ldx(X1, nV, i);
        const double l1[3] = { nextafter(q.x - r, -INFINITY), nextafter(q.y - r, -INFINITY),
                               nextafter(q.z - r, -INFINITY) };
        const double h1[3] = { nextafter(q.x + r, INFINITY), nextafter(q.y + r, INFINITY),
                               nextafter(q.z + r, INFINITY) };
#pragma unroll
        for (int k = 0; k < 3; k++) {
            lo[k] = l1[k] < lo[k] ? l1[k] : lo[k];
            hi[k] = hi[k] < h1[k] ? h1[k] : hi[k];
        }
    }
}

__global__ __launch_bounds__(BP_BLOCK) void k_mesh_aabb_partial(const double* X0,
                                                                const double* X1, int nV,
                                                                double r, double* partial)
{
    double lo[3] = { INFINITY, INFINITY, INFINITY }, hi[3] = { -INFINITY, -INFINITY, -INFINITY };
    for (int i = blockIdx.x * BP_BLOCK + threadIdx.x; i < nV; i += gridDim.x * BP_BLOCK) {
        double l[3], h[3];
        vbox(X0, X1, nV, i, r, l, h);
#pragma unroll
        for (int k = 0; k < 3; k++) {
            lo[k] = fmin(lo[k], l[k]);
            hi[k] = fmax(hi[k], h[k]);
        }
    }
#pragma unroll
    for (int k = 0; k < 3; k++)
        for (int o = 32; o > 0; o >>= 1) {
            lo[k] = fmin(lo[k], __shfl_xor(lo[k], o, WAVE));
            hi[k] = fmax(hi[k], __shfl_xor(hi[k], o, WAVE));
        }
    __shared__ double s[BP_BLOCK / WAVE][6];
    const int w = threadIdx.x / WAVE;
    if (threadIdx.x % WAVE == 0)
#pragma unroll
        for (int k = 0; k < 3; k++) {
            s[w][k] = lo[k];
            s[w][3 + k] = hi[k];
        }
    __syncthreads();
    if (threadIdx.x < 6) {
        double v = s[0][threadIdx.x];
        for (int j = 1; j < BP_BLOCK / WAVE; j++)
            v = threadIdx.x < 3 ? fmin(v, s[j][threadIdx.x]) : fmax(v, s[j][threadIdx.x]);
        partial[blockIdx.x * 6 + threadIdx.x] = v;
    }
}

__global__ __launch_bounds__(BP_BLOCK) void k_mesh_aabb_final(const double* partial, int nb,
                                                              double* aabb)
{
    __shared__ double s[BP_BLOCK / WAVE][6];
    const int w = threadIdx.x / WAVE;
#pragma unroll
    for (int k = 0; k < 6; k++) {
        double v = k < 3 ? INFINITY : -INFINITY;
        for (int j = threadIdx.x; j < nb; j += BP_BLOCK)
            v = k < 3 ? fmin(v, partial[j * 6 + k]) : fmax(v, partial[j * 6 + k]);
        for (int o = 32; o > 0; o >>= 1) {
            const double y = __shfl_xor(v, o, WAVE);
            v = k < 3 ? fmin(v, y) : fmax(v, y);
        }
        if (threadIdx.x % WAVE == 0) s[w][k] = v;
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        double v = s[0][threadIdx.x];
        for (int j = 1; j < BP_BLOCK / WAVE; j++)
            v = threadIdx.x < 3 ? fmin(v, s[j][threadIdx.x]) : fmax(v, s[j][threadIdx.x]);
        aabb[threadIdx.x] = v;
    }
}

// Batched contexts: scene boxes in two steps: workgroup (scene, chunk) reduces every
// SCENE_CHUNKS-th stretch of the scene's vertices into a partial box, then a
// lane per scene combines its partials (min / max are exact, so the box is
// the one the scene alone gets).
constexpr int SCENE_CHUNKS = 16;

__global__ __launch_bounds__(BP_BLOCK) void k_scene_aabb(const double* X0, const double* X1,
                                                         int nV, const int64_t* voff, double r,
                                                         double* part)
{
    const int sc = blockIdx.x / SCENE_CHUNKS, ch = blockIdx.x % SCENE_CHUNKS;
    double* aabb = part + 6 * (int64_t)ch; // this chunk's partial of scene sc
    double lo[3] = { INFINITY, INFINITY, INFINITY }, hi[3] = { -INFINITY, -INFINITY, -INFINITY };
    for (int64_t i = voff[sc] + (int64_t)ch * BP_BLOCK + threadIdx.x; i < voff[sc + 1];
         i += (int64_t)SCENE_CHUNKS * BP_BLOCK) {
        double l[3], h[3];
        vbox(X0, X1, nV, (int)i, r, l, h);
#pragma unroll
        for (int k = 0; k < 3; k++) {
            lo[k] = fmin(lo[k], l[k]);
            hi[k] = fmax(hi[k], h[k]);
        }
    }
#pragma unroll
    for (int k = 0; k < 3; k++)
        for (int o = 32; o > 0; o >>= 1) {
            lo[k] = fmin(lo[k], __shfl_xor(lo[k], o, WAVE));
            hi[k] = fmax(hi[k], __shfl_xor(hi[k], o, WAVE));
        }
    __shared__ double sm[BP_BLOCK / WAVE][6];
    const int w = threadIdx.x / WAVE;
    if (threadIdx.x % WAVE == 0)
#pragma unroll
        for (int k = 0; k < 3; k++) {
            sm[w][k] = lo[k];
            sm[w][3 + k] = hi[k];
        }
    __syncthreads();
    if (threadIdx.x < 6) {
        double v = sm[0][threadIdx.x];
        for (int j = 1; j < BP_BLOCK / WAVE; j++)
            v = threadIdx.x < 3 ? fmin(v, sm[j][threadIdx.x]) : fmax(v, sm[j][threadIdx.x]);
        aabb[6 * (int64_t)SCENE_CHUNKS * sc + threadIdx.x] = v;
    }
}

__global__ void k_scene_aabb_final(const double* part, int n_scenes, double* aabb)
{
    const int sc = blockIdx.x * 64 + threadIdx.x;
    if (sc >= n_scenes) return;
    const double* p = part + 6 * (int64_t)SCENE_CHUNKS * sc;
    for (int k = 0; k < 6; k++) {
        double v = p[k];
        for (int c = 1; c < SCENE_CHUNKS; c++)
            v = k < 3 ? fmin(v, p[6 * c + k]) : fmax(v, p[6 * c + k]);
        aabb[6 * (int64_t)sc + k] = v;
    }
}

__device__ __forceinline__ uint64_t expand_bits_2(uint64_t v)
{
    v = (v | v << 32) & 0x1F00000000FFFFull;
    v = (v | v << 16) & 0x1F0000FF0000FFull;
    v = (v | v << 8) & 0x100F00F00F00F00Full;
    v = (v | v << 4) & 0x10C30C30C30C30C3ull;
    v = (v | v << 2) & 0x1249249249249249ull;
    return v;
}

__device__ __forceinline__ uint64_t morton3(double x, double y, double z)
{
    const double scale = 2097152.0, top = scale - 1;
    x = x * scale;
    y = y * scale;
    z = z * scale;
    x = x < 0.0 ? 0.0 : (top < x ? top : x);
    y = y < 0.0 ? 0.0 : (top < y ? top : y);
    z = z < 0.0 ? 0.0 : (top < z ? top : z);
    return (expand_bits_2((uint64_t)x) << 2) | (expand_bits_2((uint64_t)y) << 1)
        | expand_bits_2((uint64_t)z);
}

// The trees of one broad phase as the kernels see them: every build kernel
// runs over all of them in one launch, a range of workgroups per tree.
struct TreeArgs {
    const int32_t* I;       // vertex ids per primitive (arity 1, null: all vertices)
    const int32_t* out_ids; // mesh id of each primitive (null: its index)
    int32_t n, arity;
    bool nodes;             // build the hierarchy (else only the order)
    float* box;
    uint64_t* keys;
    uint32_t* ids;
    uint64_t* mort;         // forest: copy of the codes; else null
    int32_t* lscene;        // forest: scene per sorted leaf; else null
    int4* leaf;
    Node* node;
    uint32_t *parent, *lparent; // per internal node, per sorted leaf
    int32_t* visits;
    int32_t* root;
    int32_t* front;         // refit: complete node per boundary, -1: none yet
    unsigned group0;        // first workgroup of this launch
};
constexpr int TREES = 5;
struct TreeSet {
    TreeArgs t[TREES];
    int n;
};

__device__ __forceinline__ const TreeArgs& tree_of_group(const TreeSet& S)
{
    int q = 0;
    while (q + 1 < S.n && blockIdx.x >= S.t[q + 1].group0) q++;
    return S.t[q];
}

__device__ __forceinline__ int first_vertex(const TreeArgs& T, int p)
{
    return T.I ? T.I[(int64_t)T.arity * p] : p;
}

// per primitive: FP64 box, Morton code, FP32 box.  vscene (batched contexts):
// scene per vertex, each primitive mapped by its own scene's box
__global__ __launch_bounds__(BP_BLOCK) void k_prim_boxes(TreeSet S, const double* X0,
                                                         const double* X1, int nV, double r,
                                                         const double* aabb,
                                                         const int32_t* vscene)
{
    const TreeArgs& T = tree_of_group(S);
    const int p = (blockIdx.x - T.group0) * BP_BLOCK + threadIdx.x;
    if (p >= T.n) return;
    double lo[3], hi[3];
    const int v0 = first_vertex(T, p);
    if (vscene) aabb += 6 * (int64_t)vscene[v0];
    vbox(X0, X1, nV, v0, r, lo, hi);
#pragma unroll
    for (int j = 1; j < 3; j++) {
        if (j >= T.arity) continue;
        double l[3], h[3];
        vbox(X0, X1, nV, T.I[(int64_t)T.arity * p + j], r, l, h);
#pragma unroll
        for (int k = 0; k < 3; k++) {
            lo[k] = l[k] < lo[k] ? l[k] : lo[k];
            hi[k] = hi[k] < h[k] ? h[k] : hi[k];
        }
    }
    double m[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const double c = 0.5 * (lo[k] + hi[k]);
        m[k] = (c - aabb[k]) / (aabb[3 + k] - aabb[k]);
    }
    const uint64_t code = morton3(m[0], m[1], m[2]);
    T.keys[p] = code;
    if (T.mort) T.mort[p] = code;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        T.box[(int64_t)6 * p + k] = nextafterf(__double2float_rn(lo[k]), -INFINITY);
        T.box[(int64_t)6 * p + 3 + k] = nextafterf(__double2float_rn(hi[k]), INFINITY);
    }
}

// Forest of a batched context: after the Morton sort, the scene of each
// sorted primitive becomes the key of a second stable sort (primitives of
// one scene keep their Morton order); then the Morton codes are gathered
// back in the final order and the scene of every leaf is kept.
__global__ __launch_bounds__(BP_BLOCK) void k_scene_keys(TreeSet S, const int32_t* vscene)
{
    const TreeArgs& T = tree_of_group(S);
    const int i = (blockIdx.x - T.group0) * BP_BLOCK + threadIdx.x;
    if (i < T.n) T.keys[i] = (uint64_t)vscene[first_vertex(T, (int)T.ids[i])];
}

__global__ __launch_bounds__(BP_BLOCK) void k_forest_keys(TreeSet S)
{
    const TreeArgs& T = tree_of_group(S);
    const int i = (blockIdx.x - T.group0) * BP_BLOCK + threadIdx.x;
    if (i >= T.n) return;
    T.lscene[i] = (int32_t)T.keys[i];
    T.keys[i] = T.mort[T.ids[i]];
}

// Root entry per scene before the refit: none, a single leaf, or to be
// completed (loff: the scene's first sorted leaf position, n_scenes + 1).
__global__ void k_forest_roots(const int64_t* loff, int n_scenes, int32_t* root)
{
    const int sc = blockIdx.x * 256 + threadIdx.x;
    if (sc >= n_scenes) return;
    const int64_t m = loff[sc + 1] - loff[sc];
    root[sc] = m == 0 ? ROOT_NONE : (m == 1 ? ~(int32_t)loff[sc] : ROOT_UNFINISHED);
}

// Common-prefix length of the sorted keys i and j extended by their
// positions, so equal Morton codes still order strictly; -1 outside [0, n)
// and, in a forest, across scenes (lscene: scene per sorted leaf).
__device__ __forceinline__ int delta(const uint64_t* codes, const int32_t* lscene, int n, int i,
                                     int j)
{
    if (j < 0 || j >= n) return -1;
    if (lscene && lscene[i] != lscene[j]) return -1;
    const uint64_t ci = codes[i], cj = codes[j];
    if (ci == cj) return 64 + __clz((unsigned)(i ^ j));
    return __clzll(ci ^ cj);
}

// Hierarchy of the binary radix tree over the sorted keys (Karras 2012):
// internal node i covers a key range that has i as one end and splits it at
// the highest differing bit.  Every node is placed independently, so the
// build needs no inter-thread communication.  The tree shape differs from
// the reference's Apetrei construction (lbvh.cpp:197-302); the candidate set
// does not depend on it.
//
// In a forest (lscene non-null) the prefix is -1 across scenes, so every
// scene's leaves form a tree of their own: internal node i exists when
// leaves i and i + 1 belong to one scene, and the node at a scene's first
// leaf is its root.

// Bottom-up box refit in three steps.  A workgroup owns RB_LEAVES
// consecutive leaves and completes every node whose leaves are all its own: a
// thread per leaf climbs, the first child to arrive at a node leaves its box,
// the second goes on with the union.  Every split between two such ranges
// (a boundary) belongs to one node; once its children are complete it waits
// in front[boundary].  The second step's workgroups own RB_WIDE ranges and
// climb from the boundaries inside, the third climbs from the rest in one
// workgroup.  A node is completed in the first step that owns all of its
// leaves, so boxes either come from an earlier launch or from the same
// workgroup: no inter-workgroup fences.
// Trees of two 64 x 64 sheets (24 K edges, 16 K faces): 34 launches, two
// host reads and 0.24 ms with a launch per level, 0.05 ms with these; 8 x
// 512 x 512 sheets (6.3 M edges, 4.2 M faces) 2.3 -> 1.2 ms.
constexpr int RF_BLOCK = 1024;
constexpr int RB_LEAVES = RF_BLOCK;
constexpr int RB_WIDE = 64;
constexpr int RC_BLOCK = 256; // second and third step

// A child's link to its parent i: 8 i + 4 (right child) + 2 (node i crosses
// the second step's ranges) + 1 (the first step's).
constexpr uint32_t LINK_NEAR = 1u, LINK_WIDE = 2u, LINK_RIGHT = 4u;
constexpr int LINK_SHIFT = 3;
constexpr uint32_t NO_PARENT = 0xFFFFFFFFu;
constexpr int64_t MAX_LEAVES = (1ll << 29) - 1;

__device__ __forceinline__ void write_child(Node* P, bool right, const float* lo, const float* hi)
{
    float* const l = right ? P->lo1 : P->lo0;
    float* const h = right ? P->hi1 : P->hi0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        l[k] = lo[k];
        h[k] = hi[k];
    }
}

// A thread per sorted leaf: its leaf record, and internal node i (between
// leaves i and i + 1).
__global__ __launch_bounds__(BP_BLOCK) void k_karras(TreeSet S)
{
    const TreeArgs& T = tree_of_group(S);
    const int i = (blockIdx.x - T.group0) * BP_BLOCK + threadIdx.x;
    const int n = T.n;
    if (i >= n) return;
    if (i % RB_LEAVES == 0) T.front[i / RB_LEAVES] = -1;
    { // leaf record: mesh id of the primitive and its vertices
        const int p = (int)T.ids[i];
        int v[3] = { -1, -1, -1 };
#pragma unroll
        for (int j = 0; j < 3; j++)
            if (j < T.arity) v[j] = T.I ? T.I[(int64_t)T.arity * p + j] : p;
        T.leaf[i] = make_int4(T.out_ids ? T.out_ids[p] : p, v[0], v[1], v[2]);
    }
    const uint64_t* const codes = T.keys;
    const int32_t* const lscene = T.lscene;
    const bool next = i + 1 < n && !(lscene && lscene[i] != lscene[i + 1]);
    const bool before = i > 0 && !(lscene && lscene[i - 1] != lscene[i]);
    if (!next && !before) T.lparent[i] = NO_PARENT; // the only leaf of its tree
    if (!lscene && n == 1) T.root[0] = -1; // lbvh.cpp:386-396
    if (!next) return;                     // no node between scenes
    const int d = delta(codes, lscene, n, i, i + 1) - delta(codes, lscene, n, i, i - 1) >= 0 ? 1 : -1;
    const int dmin = delta(codes, lscene, n, i, i - d);
    int lmax = 2;
    while (delta(codes, lscene, n, i, i + lmax * d) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (delta(codes, lscene, n, i, i + (l + t) * d) > dmin) l += t;
    const int j = i + l * d;
    const int dnode = delta(codes, lscene, n, i, j);
    int sp = 0;
    for (int t = (l + 1) >> 1;; t = (t + 1) >> 1) {
        if (delta(codes, lscene, n, i, i + (sp + t) * d) > dnode) sp += t;
        if (t == 1) break;
    }
    const int g = i + sp * d + (d < 0 ? -1 : 0);
    const int lo = i < j ? i : j, hi = i < j ? j : i;
    constexpr int WIDE = RB_LEAVES * RB_WIDE;
    const uint32_t link = ((uint32_t)i << LINK_SHIFT)
        | (lo / RB_LEAVES != hi / RB_LEAVES ? LINK_NEAR : 0u) | (lo / WIDE != hi / WIDE ? LINK_WIDE : 0u);
    Node* N = T.node + i;
    if (lo == g) {
        N->c0 = ~g;
        T.lparent[g] = link;
    } else {
        N->c0 = g;
        T.parent[g] = link;
    }
    if (hi == g + 1) {
        N->c1 = ~(g + 1);
        T.lparent[g + 1] = link | LINK_RIGHT;
    } else {
        N->c1 = g + 1;
        T.parent[g + 1] = link | LINK_RIGHT;
    }
    N->r0 = g;
    N->r1 = hi;
    T.visits[i] = 0;
    if (!before) { // the first leaf's node: the root
        T.parent[i] = NO_PARENT;
        T.root[lscene ? lscene[i] : 0] = ROOT_UNFINISHED;
    }
}

// A child of a node that a later step completes: with both children there,
// the node of a boundary waits in its slot (others are reached by climbing).
__device__ __forceinline__ void arrive_far(const TreeArgs& T, int32_t p)
{
    if (atomicAdd(T.visits + p, 1) == 1) T.front[T.node[p].r0 / RB_LEAVES] = p;
}

__global__ __launch_bounds__(RF_BLOCK) void k_refit_local(TreeSet S)
{
    __shared__ float sbox[RB_LEAVES][2][6]; // both children's boxes per node
    __shared__ uint32_t arrived[RB_LEAVES];
    const TreeArgs& T = tree_of_group(S);
    const int base = (int)(blockIdx.x - T.group0) * RB_LEAVES;
    const int i = base + (int)threadIdx.x;
    arrived[threadIdx.x] = 0;
    __syncthreads();
    uint32_t link = i < T.n ? T.lparent[i] : NO_PARENT;
    float lo[3] = { 0, 0, 0 }, hi[3] = { 0, 0, 0 };
    if (link != NO_PARENT) {
        const int64_t b = (int64_t)6 * T.ids[i];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            lo[k] = T.box[b + k];
            hi[k] = T.box[b + 3 + k];
        }
    }
    while (link != NO_PARENT) { // one level up per step
        const int32_t p = (int32_t)(link >> LINK_SHIFT);
        const int side = (link & LINK_RIGHT) ? 1 : 0;
        write_child(T.node + p, side != 0, lo, hi);
        if (link & LINK_NEAR) { // crosses: a later step's
            arrive_far(T, p);
            break;
        }
        float* const mine = sbox[p - base][side];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            mine[k] = lo[k];
            mine[3 + k] = hi[k];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        const uint32_t first = atomicAdd(&arrived[p - base], 1u);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        if (first == 0) break; // the other child goes on
        const float* const other = sbox[p - base][1 - side];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            lo[k] = fminf(lo[k], other[k]);
            hi[k] = fmaxf(hi[k], other[3 + k]);
        }
        link = T.parent[p];
        if (link == NO_PARENT) T.root[T.lscene ? T.lscene[p] : 0] = p; // the tree is complete
    }
}

// Climbs from the boundaries of a workgroup's ranges: `wide` boundaries
// inside every RB_WIDE ranges (the second step), else every boundary that is
// still waiting (the third, one workgroup per tree).
__global__ __launch_bounds__(RC_BLOCK) void k_refit_climb(TreeSet S, bool wide)
{
    const TreeArgs& T = tree_of_group(S);
    const int ranges = (T.n + RB_LEAVES - 1) / RB_LEAVES;
    if (wide && ranges <= RB_WIDE) return; // one group: the third step's
    const int b0 = wide ? (int)(blockIdx.x - T.group0) * RB_WIDE : 0;
    const int b1 = wide ? min(b0 + RB_WIDE - 1, ranges - 1) : ranges - 1;
    // the second step has been through the boundaries inside its ranges
    const int step = !wide && ranges > RB_WIDE ? RB_WIDE : 1;
    for (int t = (int)threadIdx.x; b0 + (t + 1) * step - 1 < b1; t += RC_BLOCK) {
        int32_t j = T.front[b0 + (t + 1) * step - 1];
        while (j >= 0) { // node j is complete
            const Node* N = T.node + j;
            float lo[3], hi[3];
#pragma unroll
            for (int k = 0; k < 3; k++) {
                lo[k] = fminf(N->lo0[k], N->lo1[k]);
                hi[k] = fmaxf(N->hi0[k], N->hi1[k]);
            }
            const uint32_t link = T.parent[j];
            if (link == NO_PARENT) {
                T.root[T.lscene ? T.lscene[j] : 0] = j; // the tree is complete
                break;
            }
            const int32_t p = (int32_t)(link >> LINK_SHIFT);
            write_child(T.node + p, (link & LINK_RIGHT) != 0, lo, hi);
            if (wide && (link & LINK_WIDE)) {
                arrive_far(T, p);
                break;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            const int32_t first = atomicAdd(T.visits + p, 1);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
            j = first == 1 ? p : -1; // else the other child goes on
        }
    }
}

__device__ __forceinline__ bool overlap(const float* q, const float* lo, const float* hi)
{
    return q[0] <= hi[0] && q[1] <= hi[1] && q[2] <= hi[2] && lo[0] <= q[3] && lo[1] <= q[4]
        && lo[2] <= q[5];
}

// CollisionMesh::can_collide as data: the intersection of the vertex
// patches filter (patch[i] != patch[j]), the static obstacle filter (i or j
// below n_dynamic) and the codim cross filter (exactly one of i, j below
// n_codim), each optional (collision_filter.hpp:113-143).
struct Filter {
    const int32_t* E;
    const int32_t* F;
    const int32_t* patch; // may be null
    int32_t n_dynamic;    // < 0: no static obstacle filter
    int32_t n_codim;      // < 0: no codim cross filter
    __device__ __forceinline__ bool any() const
    {
        return patch != nullptr || n_dynamic >= 0 || n_codim >= 0;
    }
};

__device__ __forceinline__ bool can_vv(const Filter& f, int a, int b)
{
    return (f.patch == nullptr || f.patch[a] != f.patch[b])
        && (f.n_dynamic < 0 || a < f.n_dynamic || b < f.n_dynamic)
        && (f.n_codim < 0 || ((a < f.n_codim) != (b < f.n_codim)));
}

// lbvh.cpp:826-849 can_edges_collide
__device__ __forceinline__ bool can_ee(const Filter& f, int ea, int eb)
{
    const int a0 = f.E[2 * (int64_t)ea], a1 = f.E[2 * (int64_t)ea + 1];
    const int b0 = f.E[2 * (int64_t)eb], b1 = f.E[2 * (int64_t)eb + 1];
    if (a0 == b0 || a0 == b1 || a1 == b0 || a1 == b1) return false;
    return can_vv(f, a0, b0) || can_vv(f, a0, b1) || can_vv(f, a1, b0) || can_vv(f, a1, b1);
}

// lbvh.cpp:851-858 can_face_vertex_collide
__device__ __forceinline__ bool can_fv(const Filter& f, int fi, int vi)
{
    const int f0 = f.F[3 * (int64_t)fi], f1 = f.F[3 * (int64_t)fi + 1],
              f2 = f.F[3 * (int64_t)fi + 2];
    if (vi == f0 || vi == f1 || vi == f2) return false;
    return can_vv(f, vi, f0) || can_vv(f, vi, f1) || can_vv(f, vi, f2);
}

// One lane per query leaf (in the query set's Morton order).  MODE:
//  TR_EE  edge-edge self traversal: (query, other) for other at a later
//         sorted position;
//  TR_FV  vertex queries against the face tree: (face, vertex);
//  TR_VV  codim vertices, self traversal: (query, other) in mesh ids;
//  TR_EV  codim vertex queries against the codim-edge tree: (edge, vertex)
//         in mesh ids (candidates.cpp:65-118);
//  TR_EF  edge queries against the face tree: (edge, face)
//         (lbvh.cpp:771-784 reports the same set from face queries).
enum { TR_EE = 0, TR_FV = 1, TR_VV = 2, TR_EV = 3, TR_EF = 4 };

// The query primitive: its output id and vertices (-1 padded).
struct Query {
    int id;
    int v[3];
};

// some vertex of a may collide with some vertex of b
__device__ __forceinline__ bool patch_ok(const Filter& f, const int* a, int na, const int* b,
                                         int nb)
{
    if (!f.any()) return true;
    for (int i = 0; i < na; i++)
        for (int j = 0; j < nb; j++)
            if (can_vv(f, a[i], b[j])) return true;
    return false;
}

// lbvh.cpp:800-858 filters and the reported pair for a leaf record
template <int MODE>
__device__ __forceinline__ int2 leaf_pair(const Filter& flt, const Query& q, const int4& r)
{
    if constexpr (MODE == TR_EE) { // edge vs edge: no shared vertex
        if (q.v[0] == r.y || q.v[0] == r.z || q.v[1] == r.y || q.v[1] == r.z) return make_int2(-1, -1);
        const int b[2] = { r.y, r.z };
        return patch_ok(flt, q.v, 2, b, 2) ? make_int2(q.id, r.x) : make_int2(-1, -1);
    } else if constexpr (MODE == TR_FV) { // vertex vs face
        if (q.v[0] == r.y || q.v[0] == r.z || q.v[0] == r.w) return make_int2(-1, -1);
        const int b[3] = { r.y, r.z, r.w };
        return patch_ok(flt, q.v, 1, b, 3) ? make_int2(r.x, q.id) : make_int2(-1, -1);
    } else if constexpr (MODE == TR_VV) { // codim vertex vs codim vertex
        const int b[1] = { r.y };
        return patch_ok(flt, q.v, 1, b, 1) ? make_int2(q.id, r.x) : make_int2(-1, -1);
    } else if constexpr (MODE == TR_EF) { // edge vs face (lbvh.cpp:836-849)
        if (q.v[0] == r.y || q.v[0] == r.z || q.v[0] == r.w || q.v[1] == r.y || q.v[1] == r.z
            || q.v[1] == r.w)
            return make_int2(-1, -1);
        const int b[3] = { r.y, r.z, r.w };
        return patch_ok(flt, q.v, 2, b, 3) ? make_int2(q.id, r.x) : make_int2(-1, -1);
    } else { // codim vertex vs codim edge
        if (q.v[0] == r.y || q.v[0] == r.z) return make_int2(-1, -1);
        const int b[2] = { r.y, r.z };
        return patch_ok(flt, q.v, 1, b, 2) ? make_int2(r.x, q.id) : make_int2(-1, -1);
    }
}

// SWEPT only names the launches of the swept (CCD) broad phase apart from
// the static ones in kernel profiles; the code is the same.
// Forest of a batched context (vscene non-null): every query walks the tree
// of its own scene (root_p: one entry per scene; queries of scenes that
// `active` leaves out are skipped).
struct ForestArgs {
    const int32_t* vscene;   // scene per vertex (null: one tree, root_p[0])
    const uint8_t* active;   // per scene (null: all)
    const uint32_t* tids;    // target tree: primitive per sorted leaf
};

struct TraverseArgs {
    const float* qbox;
    const uint32_t* qids;
    int nq;
    const Node* nodes;
    const int32_t* root;
    const int4* leaf;
    const float* tbox;
    int nleaves;
    Filter flt;
    const int32_t* qmap;
    int2* out;
    Shards S;
    int* deep; // pool of `slots` spill stacks, TR_STACK - TR_LSTACK ints each
    unsigned* claimed;
    unsigned slots;
    int* status;
    ForestArgs fa;
    int qw; // queries a wave starts with (its first lanes; the others share)
};

template <int BLOCK> struct TrShared {
    int stack[TR_LSTACK][BLOCK];
    int leaf[BLOCK / WAVE][TR_QUEUE];
    unsigned char lane[BLOCK / WAVE][TR_QUEUE];
    unsigned char donor[BLOCK / WAVE][WAVE];
};

// LDS written by some lanes of the wave is read by others
__device__ __forceinline__ void wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The walk of one workgroup's queries (block: its index in the query set's
// launch range).  stack: postponed right children, the first TR_LSTACK
// entries of each lane in LDS (small enough for full occupancy); a lane that
// goes deeper claims a spill stack in HBM and keeps it.  (A spill stack per
// lane is 12 KB per wave: with 8 queries a wave, 1.5 KB per query.)
template <int MODE, int BLOCK>
__device__ __forceinline__ void traverse(const TraverseArgs& A, unsigned block,
                                         TrShared<BLOCK>& sh_mem)
{
    const float* const qbox = A.qbox;
    const uint32_t* const qids = A.qids;
    const int nq = A.nq, nleaves = A.nleaves;
    const Node* const nodes = A.nodes;
    const int32_t* const root_p = A.root;
    const int4* const leaf = A.leaf;
    const float* const tbox = A.tbox;
    const Filter& flt = A.flt;
    const int32_t* const qmap = A.qmap;
    int2* const out = A.out;
    const Shards& S = A.S;
    int* const status = A.status;
    const ForestArgs& fa = A.fa;
    int(*const stack)[BLOCK] = sh_mem.stack;
    constexpr bool TRI = MODE == TR_EE || MODE == TR_VV;
    const int t = threadIdx.x;
    const int64_t q0 = ((int64_t)block * (BLOCK / WAVE) + t / WAVE) * A.qw + t % WAVE;
    const bool has_query = t % WAVE < A.qw && q0 < nq;
    const int qpos = has_query ? (int)q0 : 0;
    bool active = has_query;
    int* deep = nullptr; // its entry TR_LSTACK is the spill stack's first
    float q[6] = { 0, 0, 0, 0, 0, 0 };
    Query qr { 0, { -1, -1, -1 } };
    if (active) {
        const int qprim = (int)qids[qpos];
#pragma unroll
        for (int k = 0; k < 6; k++) q[k] = qbox[(int64_t)6 * qprim + k];
        if (MODE == TR_EE || MODE == TR_EF) { // query edge: id, endpoints
            qr.id = qprim;
            qr.v[0] = flt.E[2 * (int64_t)qprim];
            qr.v[1] = flt.E[2 * (int64_t)qprim + 1];
        } else { // query vertex (codim queries map their subset index)
            qr.id = qmap ? qmap[qprim] : qprim;
            qr.v[0] = qr.id;
        }
    }
    const int nin = nleaves - 1; // internal nodes
    const int sh = wave_shard();
    // Overlapping leaves (position and lane) wait in the wave's queue in LDS.
    // Past half of it, or when the walks end, a lane takes every 64th entry:
    // the leaf records of all of them are loaded at once, the filters drop
    // pairs, and one append writes the rest.  (The append's round trip is the
    // dear part: with four entries held per lane the busiest lane forced one
    // every few steps, for a handful of pairs each; 11.4 against 9.4 ms for
    // the static walks of 8 sheets of 512^2.)
    int* const qleaf = sh_mem.leaf[t / WAVE];
    unsigned char* const qlane = sh_mem.lane[t / WAVE];
    unsigned nb = 0; // uniform
    int owner = t % WAVE; // lane whose query this lane walks
    auto push = [&](int h) {
        const unsigned long long m = __ballot(h >= 0);
        if (h >= 0) {
            const unsigned at = nb + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                         __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
            qleaf[at] = h;
            qlane[at] = (unsigned char)owner;
        }
        nb += (unsigned)__popcll(m);
    };
    int2* const reg = out + sh * S.scap;
    auto flush = [&]() {
        constexpr int R = TR_QUEUE / WAVE;
        wave_fence();
        int lp[R], ln[R];
#pragma unroll
        for (int k = 0; k < R; k++) {
            const unsigned i = k * WAVE + t % WAVE;
            lp[k] = i < nb ? qleaf[i] : -1;
            ln[k] = i < nb ? qlane[i] : 0;
        }
        int4 rec[R]; // every load first, then the filters
#pragma unroll
        for (int k = 0; k < R; k++) {
            rec[k] = make_int4(-1, -1, -1, -1);
            if (lp[k] >= 0) rec[k] = leaf[lp[k]];
        }
        int2 hit[R];
        unsigned before[R], total = 0;
#pragma unroll
        for (int k = 0; k < R; k++) {
            Query q2;
            q2.id = __shfl(qr.id, ln[k], WAVE);
#pragma unroll
            for (int v = 0; v < 3; v++) q2.v[v] = __shfl(qr.v[v], ln[k], WAVE);
            hit[k] = lp[k] >= 0 ? leaf_pair<MODE>(flt, q2, rec[k]) : make_int2(-1, -1);
            const unsigned long long m = __ballot(hit[k].x >= 0);
            before[k] = total + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                    __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
            total += (unsigned)__popcll(m);
        }
        if (total) {
            unsigned long long base = 0;
            if (t % WAVE == 0)
                base = atomicAdd(S.cnt + (int64_t)sh * SHARD_PAD, (unsigned long long)total);
            const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)base);
            const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(base >> 32));
            const int64_t first = (int64_t)(((unsigned long long)hi << 32) | lo);
#pragma unroll
            for (int k = 0; k < R; k++)
                if (hit[k].x >= 0 && first + before[k] < S.scap) reg[first + before[k]] = hit[k];
        }
        nb = 0;
        wave_fence();
    };
    int single = -1; // the only leaf of a one-leaf tree
    int node = 0;
    if (active) {
        int root = root_p[0];
        if (fa.vscene) {
            const int sc = fa.vscene[qr.v[0]];
            root = root_p[sc];
            if (root == ROOT_NONE || (fa.active && !fa.active[sc])) active = false;
        }
        if (!active) {
        } else if (root < -nleaves || root >= (nin > 0 ? nin : 1)) {
            // the build did not finish: refuse to walk
            atomicOr(status, 2);
            active = false;
        } else if (root < 0) { // single target leaf (lbvh.cpp:386-396)
            if (!TRI) {
                const int lp = ~root;
                const float* b = tbox + (int64_t)6 * (fa.tids ? fa.tids[lp] : 0);
                if (overlap(q, b, b + 3)) single = lp;
            }
            active = false;
        } else {
            node = root;
        }
    }
    push(single);
    // Postponed children of the lane: entries [sb, sp) (those below sb were
    // given away).  Lanes of a wave finish at different times; every
    // TR_SHARE steps the idle ones take the oldest postponed child, the
    // largest subtree left, of a busy lane each and walk it with that lane's
    // query (9.4 to 8.4 ms there, 0.29 to 0.21 ms on 4 sheets of 97^2).
    int sb = 0, sp = 0, steps = 0;
    unsigned round = 0;
    int pos = qpos; // of the query walked
    unsigned char* const donor = sh_mem.donor[t / WAVE];
    const int max_steps = 2 * nleaves + 64; // each node is visited at most once per query
    // A subtree that changes lanes starts a count of its own, so the wave's rounds
    // are bounded too: in each of them a query that started here visits a node.
    const int64_t visits = (int64_t)A.qw * max_steps;
    const unsigned max_rounds = visits < (int64_t)UINT32_MAX ? (unsigned)visits : UINT32_MAX;
    while (__any(active)) {
        if (round == max_rounds) {
            atomicOr(status, 2);
            break;
        }
        if (++round % TR_SHARE == 0) {
            const bool gives = active && sp > sb && sb < TR_LSTACK;
            const bool takes = !active;
            const unsigned long long mg = __ballot(gives), mt = __ballot(takes);
            const unsigned ng = (unsigned)__popcll(mg), nt = (unsigned)__popcll(mt);
            if (ng > 0 && nt >= TR_IDLE) {
                const unsigned long long mine = gives ? mg : mt;
                const unsigned rank = __builtin_amdgcn_mbcnt_hi((unsigned)(mine >> 32),
                                          __builtin_amdgcn_mbcnt_lo((unsigned)mine, 0u));
                if (gives) donor[rank] = (unsigned char)(t % WAVE);
                wave_fence();
                const bool got = takes && rank < ng;
                const int src = got ? donor[rank] : t % WAVE;
#pragma unroll
                for (int k = 0; k < 6; k++) {
                    const float v = __shfl(q[k], src, WAVE);
                    q[k] = got ? v : q[k];
                }
                const int pos2 = __shfl(pos, src, WAVE), own2 = __shfl(owner, src, WAVE),
                          sb2 = __shfl(sb, src, WAVE);
                if (got) {
                    pos = pos2;
                    owner = own2;
                    node = stack[sb2][t - t % WAVE + src];
                    sb = sp = steps = 0;
                    active = true;
                } else if (gives && rank < nt) {
                    sb++;
                }
                wave_fence();
            }
        }
        int h0 = -1, h1 = -1;
        bool nd_ok = true;
        if (active) {
            const Node nd = nodes[node]; // node: a valid index (checked when it was read)
            // links must name an internal node or a leaf position, and a walk
            // visits each node at most once: one rarely taken branch for both
            ++steps;
            if ((steps > max_steps) | (nd.c0 >= nin) | (nd.c1 >= nin) | (nd.c0 < -nleaves)
                | (nd.c1 < -nleaves)) {
                atomicOr(status, 2);
                active = false;
                nd_ok = false;
            }
            // branch-free tests (bitwise, no short-circuit)
            bool o0 = nd_ok & overlap(q, nd.lo0, nd.hi0), o1 = nd_ok & overlap(q, nd.lo1, nd.hi1);
            if (TRI) {
                o0 = o0 & (nd.r0 > pos);
                o1 = o1 & (nd.r1 > pos);
            }
            const bool l0 = nd.c0 < 0, l1 = nd.c1 < 0;
            h0 = (o0 & l0) ? ~nd.c0 : -1;
            h1 = (o1 & l1) ? ~nd.c1 : -1;
            const bool t0 = o0 & !l0, t1 = o1 & !l1;
            if (!nd_ok) {
            } else if (!t0 && !t1) {
                if (sp == sb) active = false;
                else {
                    --sp;
                    // the LDS entries by an LDS read; the deep ones through a
                    // load of their own (a shared select of the two addresses
                    // would turn every pop into a flat load)
                    if (sp < TR_LSTACK)
                        node = stack[sp][t];
                    else
                        node = __builtin_nontemporal_load(
                            &deep[sp]);
                }
            } else {
                node = t0 ? nd.c0 : nd.c1;
                if (t0 && t1) {
                    if (sp < TR_LSTACK) stack[sp++][t] = nd.c1;
                    else if (sp < TR_STACK) {
                        if (!deep) {
                            const unsigned k = atomicAdd(A.claimed, 1u);
                            if (k < A.slots)
                                deep = A.deep + (int64_t)k * (TR_STACK - TR_LSTACK) - TR_LSTACK;
                        }
                        if (deep) {
                            deep[sp] = nd.c1;
                            sp++;
                        } else { // the host walks again with a larger pool
                            atomicOr(status, 4);
                            active = false;
                        }
                    } else {
                        atomicOr(status, 1);
                        active = false;
                    }
                }
            }
        }
        push(h0);
        push(h1);
        if (nb > TR_QUEUE - 2 * WAVE) flush(); // room for the next step's
    }
    if (nb > 0) flush();
}

// BLOCK: workgroup size (64, 128 or 256), chosen per launch by the
// context's autotuner or TR_BLOCK.
template <int MODE, int SWEPT, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_traverse(TraverseArgs a)
{
    __shared__ TrShared<BLOCK> m;
    traverse<MODE, BLOCK>(a, xcd_block(), m);
}

// Edge-edge and face-vertex walks side by side (workgroups [0, nb_ee) and
// the rest).  Bound by the chain of dependent node loads of the longest walk
// (small scenes: two launches in a row take two of them) and by node reads
// from L2 (large ones).  With the wave's queue and the shared subtrees,
// static walks of 4 sheets of 97^2 go from 0.395 + 0.292 to 0.138 ms, of
// 8 sheets of 512^2 from 8.35 + 3.09 to 8.33 ms (vertices off the grid; 9.5 ms
// with the sheets exactly above each other).
template <int SWEPT, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_traverse_both(TraverseArgs ee, TraverseArgs fv,
                                                         unsigned nb_ee)
{
    __shared__ TrShared<BLOCK> m;
    if (blockIdx.x < nb_ee)
        traverse<TR_EE, BLOCK>(ee, xcd_block(blockIdx.x, nb_ee), m);
    else
        traverse<TR_FV, BLOCK>(fv, xcd_block(blockIdx.x - nb_ee, gridDim.x - nb_ee), m);
}

unsigned traverse_blocks(int64_t nq, int qw, int block)
{
    return grid_for(nq, block / WAVE * qw);
}

// lanes of a walk of nq queries (its largest workgroup size)
int64_t walk_lanes(int64_t nq, int qw) { return ((nq + qw - 1) / qw + 4) * WAVE; }

// The pool of spill stacks: SLOTS_MIN of them (no sheet stack, sphere row or batch of
// the benchmarks needs one), then as many as a walk has needed
// (grown by 4 when one finds it empty, at most a stack per lane).
constexpr int64_t SLOTS_MIN = 1024;
constexpr size_t SLOT_BYTES = sizeof(int) * (TR_STACK - TR_LSTACK);

unsigned reserve_slots(Ctx& c, int64_t lanes)
{
    const int64_t n = std::min(std::max(c.tr_slots, SLOTS_MIN), lanes);
    c.tr_deep.reserve(SLOT_BYTES * (size_t)n);
    return (unsigned)n;
}

// after a walk: whether it has to run again with a larger pool
bool slots_short(Ctx& c, int status, unsigned slots, int64_t lanes)
{
    if (!(status & 4)) return false;
    if (slots >= lanes) throw Error(IPCG_ERR_NUMERIC, "LBVH spill stacks ran out");
    c.tr_slots = std::min<int64_t>(4 * (int64_t)slots, lanes);
    return true;
}

// the walks' status word, then the number of spill stacks claimed
struct WalkStatus {
    int status;
    unsigned claimed;
};

// A walk of few queries leaves most of the chip idle and takes the time of
// its longest wave: its waves start with part of their lanes busy, and the
// others take over subtrees.  Static walks with 64, 16, 8 queries a wave: 0.091,
// 0.039, 0.033 ms for 33K queries (two 64^2 sheets), 0.207, 0.138, 0.141 ms for
// 149K (4 sheets of 97^2), 0.086, 0.125 ms for the 450K short walks of 11 spheres.
int wave_queries(int64_t nq) { return nq <= TR_FEWER ? 8 : nq <= TR_FEW ? 16 : WAVE; }

template <int MODE, int SWEPT, int BLOCK>
void launch_traverse_b(const TraverseArgs& a, hipStream_t s)
{
    hipLaunchKernelGGL((k_traverse<MODE, SWEPT, BLOCK>), dim3(traverse_blocks(a.nq, a.qw, BLOCK)),
                       dim3(BLOCK), 0, s, a);
}

template <int MODE, int SWEPT> void launch_traverse(int block, const TraverseArgs& a, hipStream_t s)
{
    if (block == 64) launch_traverse_b<MODE, SWEPT, 64>(a, s);
    else if (block == 256) launch_traverse_b<MODE, SWEPT, 256>(a, s);
    else launch_traverse_b<MODE, SWEPT, TR_BLOCK>(a, s);
}

template <int SWEPT, int BLOCK>
void launch_both_b(const TraverseArgs& ee, const TraverseArgs& fv, hipStream_t s)
{
    const unsigned nb_ee = traverse_blocks(ee.nq, ee.qw, BLOCK),
                   nb_fv = traverse_blocks(fv.nq, fv.qw, BLOCK);
    hipLaunchKernelGGL((k_traverse_both<SWEPT, BLOCK>), dim3(nb_ee + nb_fv), dim3(BLOCK), 0, s, ee,
                       fv, nb_ee);
}

template <int SWEPT>
void launch_both(int block, const TraverseArgs& ee, const TraverseArgs& fv, hipStream_t s)
{
    if (block == 64) launch_both_b<SWEPT, 64>(ee, fv, s);
    else if (block == 256) launch_both_b<SWEPT, 256>(ee, fv, s);
    else launch_both_b<SWEPT, TR_BLOCK>(ee, fv, s);
}

constexpr int TUNE_BLOCKS[3] = { 64, 128, 256 };

// One traversal launch with the workgroup size tuned for this context: on
// the first call of `stage` with autotuning on, every size runs once on the
// real input (its output is discarded by clearing the lists' shard counters,
// `sets` of them from cnt) and the fastest, by HIP events on the context
// stream, is kept.  Candidate sets do not depend on the size.
template <class Launch>
void tuned_traverse(Ctx& c, const std::string& stage, unsigned long long* cnt, int sets,
                    unsigned* claimed, Launch&& launch)
{
    hipStream_t s = c.stream;
    auto clear = [&]() {
        IPCG_HIP(hipMemsetAsync(cnt, 0, SHARD_CNT_BYTES * (size_t)sets, s));
        IPCG_HIP(hipMemsetAsync(claimed, 0, sizeof(unsigned), s));
    };
    auto it = c.launch_block.find(stage);
    int block = it != c.launch_block.end() ? it->second : 0;
    if (block == 0 && c.autotune) {
        hipEvent_t e0, e1;
        IPCG_HIP(hipEventCreate(&e0));
        IPCG_HIP(hipEventCreate(&e1));
        float best = INFINITY;
        for (int b : TUNE_BLOCKS) {
            clear();
            IPCG_HIP(hipEventRecord(e0, s));
            launch(b);
            IPCG_HIP(hipEventRecord(e1, s));
            IPCG_HIP(hipEventSynchronize(e1));
            float ms = 0;
            IPCG_HIP(hipEventElapsedTime(&ms, e0, e1));
            c.tune_ms[stage + "@" + std::to_string(b)] = ms;
            if (ms < best) {
                best = ms;
                block = b;
            }
        }
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        c.launch_block[stage] = block;
        clear();
    }
    launch(block ? block : TR_BLOCK);
}

// ---------------------------------------------------------------------------
// Sweep and prune (sweep_and_prune.cpp:22-249 over scalable-ccd's
// sort_and_sweep): FP64 boxes sorted by (min along the sweep axis, id); a
// lane per sorted box scans forward while the next box starts within its
// extent along the axis and reports full 3D overlaps that pass the filters.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t ordered_bits(double x)
{
    x = x + 0.0; // -0 -> +0: equal keys stay equal
    const uint64_t b = (uint64_t)__double_as_longlong(x);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}

template <int ARITY>
__global__ __launch_bounds__(BP_BLOCK) void k_sap_boxes(const double* X0, const double* X1,
                                                        int nV, const int32_t* I, int n, double r,
                                                        int axis, double* box64, uint64_t* keys)
{
    const int p = blockIdx.x * BP_BLOCK + threadIdx.x;
    if (p >= n) return;
    double lo[3], hi[3];
    vbox(X0, X1, nV, ARITY == 1 ? p : I[(int64_t)ARITY * p], r, lo, hi);
#pragma unroll
    for (int j = 1; j < ARITY; j++) {
        double l[3], h[3];
        vbox(X0, X1, nV, I[(int64_t)ARITY * p + j], r, l, h);
#pragma unroll
        for (int k = 0; k < 3; k++) {
            lo[k] = l[k] < lo[k] ? l[k] : lo[k];
            hi[k] = hi[k] < h[k] ? h[k] : hi[k];
        }
    }
#pragma unroll
    for (int k = 0; k < 3; k++) {
        box64[(int64_t)6 * p + k] = lo[k];
        box64[(int64_t)6 * p + 3 + k] = hi[k];
    }
    keys[p] = ordered_bits(lo[axis]);
}

// boxes in sorted order (coalesced sweeps)
__global__ __launch_bounds__(BP_BLOCK) void k_sap_gather(const double* box64, const uint32_t* ids,
                                                         int n, double* sorted)
{
    const int i = blockIdx.x * BP_BLOCK + threadIdx.x;
    if (i >= n) return;
    const uint32_t p = ids[i];
#pragma unroll
    for (int k = 0; k < 6; k++) sorted[(int64_t)6 * i + k] = box64[(int64_t)6 * p + k];
}

__device__ __forceinline__ bool overlap64(const double* a, const double* b)
{
    return a[0] <= b[3] && a[1] <= b[4] && a[2] <= b[5] && b[0] <= a[3] && b[1] <= a[4]
        && b[2] <= a[5];
}

// Edge-edge: pairs (earlier, later) in sorted order.
__global__ __launch_bounds__(TR_BLOCK) void k_sap_self(const double* sb, const uint32_t* ids, int n,
                                                       int axis, Filter flt, int2* out, Shards S)
{
    const int i = blockIdx.x * TR_BLOCK + threadIdx.x;
    bool active = i < n;
    double a[6] = { 0, 0, 0, 0, 0, 0 };
    int ai = 0;
    if (active) {
#pragma unroll
        for (int k = 0; k < 6; k++) a[k] = sb[(int64_t)6 * i + k];
        ai = (int)ids[i];
    }
    const int sh = wave_shard();
    int j = i + 1;
    while (__any(active)) {
        int hit = -1;
        if (active) {
            if (j >= n || sb[(int64_t)6 * j + axis] > a[3 + axis]) {
                active = false;
            } else {
                const int bj = (int)ids[j];
                if (overlap64(a, sb + (int64_t)6 * j) && can_ee(flt, ai, bj)) hit = bj;
                j++;
            }
        }
        unsigned pre;
        const int64_t slot = (int64_t)shard_append_bits(S, sh, hit >= 0, false, pre) + pre;
        if (hit >= 0 && slot < S.scap) out[sh * S.scap + slot] = make_int2(ai, hit);
    }
}

// Face-vertex from one side: each query box (sorted, `qa`) scans the other
// list (`sb`) from the first box starting at (STRICT: after) its own start.
// FACES: the queries are faces; otherwise vertices.
template <bool FACES, bool STRICT>
__global__ __launch_bounds__(TR_BLOCK) void k_sap_cross(const double* qa, const uint32_t* qids,
                                                        int nq, const double* sb,
                                                        const uint32_t* sids, int ns, int axis,
                                                        Filter flt, int2* out, Shards S)
{
    const int i = blockIdx.x * TR_BLOCK + threadIdx.x;
    bool active = i < nq;
    double a[6] = { 0, 0, 0, 0, 0, 0 };
    int ai = 0, j = 0;
    if (active) {
#pragma unroll
        for (int k = 0; k < 6; k++) a[k] = qa[(int64_t)6 * i + k];
        ai = (int)qids[i];
        int lo = 0, hi = ns;
        while (lo < hi) {
            const int m = (lo + hi) >> 1;
            const double km = sb[(int64_t)6 * m + axis];
            if (STRICT ? km <= a[axis] : km < a[axis]) lo = m + 1;
            else hi = m;
        }
        j = lo;
    }
    const int sh = wave_shard();
    while (__any(active)) {
        int2 hit = make_int2(-1, -1);
        if (active) {
            if (j >= ns || sb[(int64_t)6 * j + axis] > a[3 + axis]) {
                active = false;
            } else {
                const int bj = (int)sids[j];
                const int f = FACES ? ai : bj, v = FACES ? bj : ai;
                if (overlap64(a, sb + (int64_t)6 * j) && can_fv(flt, f, v)) hit = make_int2(f, v);
                j++;
            }
        }
        unsigned pre;
        const int64_t slot = (int64_t)shard_append_bits(S, sh, hit.x >= 0, false, pre) + pre;
        if (hit.x >= 0 && slot < S.scap) out[sh * S.scap + slot] = hit;
    }
}

// A tree to build (or, without nodes, an order): the primitives of a set
struct TreeJob {
    Tree* T;
    const int32_t* I;
    int arity;
    int n;
    bool nodes;
    const int32_t* out_ids;            // mesh id of each primitive (null: its index)
    const std::vector<int64_t>* loff;  // batched contexts: each scene's first primitive
};

// the sets of one broad phase sorted along an axis (FP64 boxes)
void sap_lists(Ctx& c, const TreeJob* jobs, int nj, const double* X0, const double* X1, double r,
               int axis)
{
    hipStream_t s = c.stream;
    SortJob sj[TREES];
    int ns = 0;
    for (int q = 0; q < nj; q++) {
        Tree& T = *jobs[q].T;
        const int n = jobs[q].n;
        T.n = n;
        if (n <= 0) continue;
        T.box.reserve(sizeof(double) * 6 * (size_t)n);
        T.sbox.reserve(sizeof(double) * 6 * (size_t)n);
        T.keys.reserve(sizeof(uint64_t) * (size_t)n);
        T.keys2.reserve(sizeof(uint64_t) * (size_t)n);
        T.ids.reserve(sizeof(uint32_t) * (size_t)n);
        T.ids2.reserve(sizeof(uint32_t) * (size_t)n);
        const unsigned g = grid_for(n, BP_BLOCK);
        const auto k = jobs[q].arity == 1 ? k_sap_boxes<1>
            : jobs[q].arity == 2          ? k_sap_boxes<2>
                                          : k_sap_boxes<3>;
        hipLaunchKernelGGL(k, dim3(g), dim3(BP_BLOCK), 0, s, X0, X1, c.nV, jobs[q].I, n, r, axis,
                           T.box.as<double>(), T.keys.as<uint64_t>());
        IPCG_CHECK_LAUNCH();
        sj[ns++] = { T.keys.p, T.keys2.p, T.ids.as<uint32_t>(), T.ids2.as<uint32_t>(), n, ~0ull,
                     true, false };
    }
    radix_sort_jobs(c.sort_space, sj, ns, s);
    ns = 0;
    for (int q = 0; q < nj; q++) {
        Tree& T = *jobs[q].T;
        if (T.n <= 0) continue;
        if (sj[ns++].in_alt) {
            std::swap(T.keys, T.keys2);
            std::swap(T.ids, T.ids2);
        }
        hipLaunchKernelGGL(k_sap_gather, dim3(grid_for(T.n, BP_BLOCK)), dim3(BP_BLOCK), 0, s,
                           T.box.as<double>(), T.ids.as<uint32_t>(), T.n, T.sbox.as<double>());
        IPCG_CHECK_LAUNCH();
    }
}

// LBVHs of the sets of one broad phase.  Batched contexts build forests:
// primitives of a scene are contiguous, c.vscene is the scene per vertex.
void build_trees(Ctx& c, const TreeJob* jobs, int nj, const double* X0, const double* X1, double r)
{
    hipStream_t s = c.stream;
    const bool forest = c.batched();
    const int S = forest ? c.n_scenes : 1;
    const int32_t* vscene = forest ? c.vscene.as<int32_t>() : nullptr;
    TreeSet all {}; // trees with primitives
    Tree* of[TREES];
    SortJob sj[TREES];
    // first workgroup of each tree for launches of `per` primitives a workgroup
    auto groups = [](TreeSet& set, int per) {
        unsigned at = 0;
        for (int q = 0; q < set.n; q++) {
            set.t[q].group0 = at;
            at += grid_for(set.t[q].n, per);
        }
        return at;
    };
    for (int q = 0; q < nj; q++) {
        const TreeJob& J = jobs[q];
        Tree& T = *J.T;
        T.n = J.n;
        T.root.reserve(sizeof(int32_t) * (size_t)S);
        if (forest) { // root entries for scenes with no or one primitive
            T.loff.reserve(sizeof(int64_t) * J.loff->size());
            // (the vectors live as long as the mesh)
            IPCG_HIP(hipMemcpyAsync(T.loff.p, J.loff->data(), sizeof(int64_t) * J.loff->size(),
                                    hipMemcpyHostToDevice, s));
            hipLaunchKernelGGL(k_forest_roots, dim3(grid_for(S, 256)), dim3(256), 0, s,
                               T.loff.as<int64_t>(), S, T.root.as<int32_t>());
            IPCG_CHECK_LAUNCH();
        }
        const size_t n = (size_t)std::max(J.n, 0);
        if (n == 0) continue;
        if ((int64_t)n > MAX_LEAVES) throw Error(IPCG_ERR_ARG, "too many primitives for an LBVH");
        T.box.reserve(sizeof(float) * 6 * n);
        T.keys.reserve(sizeof(uint64_t) * n);
        T.keys2.reserve(sizeof(uint64_t) * n);
        T.ids.reserve(sizeof(uint32_t) * n);
        T.ids2.reserve(sizeof(uint32_t) * n);
        if (forest) {
            T.mort.reserve(sizeof(uint64_t) * n);
            T.lscene.reserve(sizeof(int32_t) * n);
        }
        TreeArgs a {};
        a.I = J.I;
        a.out_ids = J.out_ids;
        a.n = J.n;
        a.arity = J.arity;
        a.nodes = J.nodes;
        a.root = T.root.as<int32_t>();
        if (J.nodes) {
            T.leaf.reserve(sizeof(int4) * n);
            T.nodes.reserve(sizeof(Node) * (n > 1 ? n - 1 : 1));
            // int32 arrays of n: parent, lparent, visits; front
            T.info.reserve(sizeof(int32_t) * (3 * n + n / RB_LEAVES + 1));
            a.leaf = T.leaf.as<int4>();
            a.node = T.nodes.as<Node>();
            a.parent = T.info.as<uint32_t>();
            a.lparent = a.parent + n;
            a.visits = reinterpret_cast<int32_t*>(a.lparent + n);
            a.front = a.visits + n;
        }
        of[all.n] = &T;
        all.t[all.n++] = a;
    }
    if (all.n == 0) return;
    auto buffers = [&]() { // after the sorts' ping-pong
        for (int q = 0; q < all.n; q++) {
            all.t[q].box = of[q]->box.as<float>();
            all.t[q].keys = of[q]->keys.as<uint64_t>();
            all.t[q].ids = of[q]->ids.as<uint32_t>();
            all.t[q].mort = forest ? of[q]->mort.as<uint64_t>() : nullptr;
            all.t[q].lscene = forest ? of[q]->lscene.as<int32_t>() : nullptr;
        }
    };
    auto sort = [&](unsigned long long mask, bool iota) {
        for (int q = 0; q < all.n; q++)
            sj[q] = { of[q]->keys.p, of[q]->keys2.p, of[q]->ids.as<uint32_t>(),
                      of[q]->ids2.as<uint32_t>(), all.t[q].n, mask, iota, false };
        radix_sort_jobs(c.sort_space, sj, all.n, s);
        for (int q = 0; q < all.n; q++)
            if (sj[q].in_alt) {
                std::swap(of[q]->keys, of[q]->keys2);
                std::swap(of[q]->ids, of[q]->ids2);
            }
        buffers();
    };
    buffers();
    const unsigned g = groups(all, BP_BLOCK);
    hipLaunchKernelGGL(k_prim_boxes, dim3(g), dim3(BP_BLOCK), 0, s, all, X0, X1, c.nV, r,
                       c.aabb.as<double>(), vscene);
    IPCG_CHECK_LAUNCH();
    c.stage_begin("bp_sort");
    sort(low_bits(63), true);
    if (forest) { // stable second pass by scene, then the Morton codes in that order
        hipLaunchKernelGGL(k_scene_keys, dim3(g), dim3(BP_BLOCK), 0, s, all, vscene);
        IPCG_CHECK_LAUNCH();
        int bits = 1;
        while ((1ll << bits) < S) bits++;
        sort(low_bits(bits), false);
        hipLaunchKernelGGL(k_forest_keys, dim3(g), dim3(BP_BLOCK), 0, s, all);
        IPCG_CHECK_LAUNCH();
    }
    c.stage_end();
    TreeSet trees {};
    for (int q = 0; q < all.n; q++)
        if (all.t[q].nodes) trees.t[trees.n++] = all.t[q];
    if (trees.n == 0) return;
    c.stage_begin("bp_build");
    const unsigned gk = groups(trees, BP_BLOCK);
    hipLaunchKernelGGL(k_karras, dim3(gk), dim3(BP_BLOCK), 0, s, trees);
    const unsigned gl = groups(trees, RB_LEAVES);
    hipLaunchKernelGGL(k_refit_local, dim3(gl), dim3(RF_BLOCK), 0, s, trees);
    IPCG_CHECK_LAUNCH();
    int most = 0;
    for (int q = 0; q < trees.n; q++) most = std::max(most, trees.t[q].n);
    if (most > RB_LEAVES * RB_WIDE) {
        const unsigned gw = groups(trees, RB_LEAVES * RB_WIDE);
        hipLaunchKernelGGL(k_refit_climb, dim3(gw), dim3(RC_BLOCK), 0, s, trees, true);
    }
    if (most > RB_LEAVES) {
        for (int q = 0; q < trees.n; q++) trees.t[q].group0 = (unsigned)q;
        hipLaunchKernelGGL(k_refit_climb, dim3(trees.n), dim3(RC_BLOCK), 0, s, trees, false);
    }
    IPCG_CHECK_LAUNCH();
    c.stage_end();
}

ForestArgs forest_args(const Ctx& c, const Tree& target)
{
    if (!c.batched()) return { nullptr, nullptr, target.ids.as<uint32_t>() };
    return { c.vscene.as<int32_t>(), c.all_active ? nullptr : c.scene_active.as<uint8_t>(),
             target.ids.as<uint32_t>() };
}

// mesh box of the vertex boxes (broad_phase.cpp:93-125) into c.aabb
void mesh_bounds(Ctx& c, const double* X0, const double* X1, double inflation)
{
    hipStream_t s = c.stream;
    c.stage_begin("bp_boxes");
    if (c.batched()) { // one box per scene
        c.aabb.reserve(sizeof(double) * 6 * (size_t)c.n_scenes);
        c.aabb_partial.reserve(sizeof(double) * 6 * SCENE_CHUNKS * (size_t)c.n_scenes);
        hipLaunchKernelGGL(k_scene_aabb, dim3(SCENE_CHUNKS * c.n_scenes), dim3(BP_BLOCK), 0, s, X0,
                           X1, c.nV, c.voff_d.as<int64_t>(), inflation,
                           c.aabb_partial.as<double>());
        hipLaunchKernelGGL(k_scene_aabb_final, dim3((c.n_scenes + 63) / 64), dim3(64), 0, s,
                           c.aabb_partial.as<double>(), c.n_scenes, c.aabb.as<double>());
        IPCG_CHECK_LAUNCH();
        c.stage_end();
        return;
    }
    const int nb = (int)grid_for(c.nV, BP_BLOCK, 1024);
    c.aabb_partial.reserve(sizeof(double) * 6 * nb);
    c.aabb.reserve(sizeof(double) * 6);
    hipLaunchKernelGGL(k_mesh_aabb_partial, dim3(nb), dim3(BP_BLOCK), 0, s, X0, X1, c.nV,
                       inflation, c.aabb_partial.as<double>());
    hipLaunchKernelGGL(k_mesh_aabb_final, dim3(1), dim3(BP_BLOCK), 0, s, c.aabb_partial.as<double>(),
                       nb, c.aabb.as<double>());
    IPCG_CHECK_LAUNCH();
    c.stage_end();
}

} // namespace

void bp_build(Ctx& c, bool swept, double inflation, int method)
{
    c.require_mesh();
    c.require_pos(0);
    if (swept) c.require_pos(1);
    if (method != IPCG_BP_LBVH && method != IPCG_BP_SAP)
        throw Error(IPCG_ERR_ARG, "unsupported broad phase method");
    const bool sap = method == IPCG_BP_SAP;
    if (sap && c.batched())
        throw Error(IPCG_ERR_ARG, "a batched context supports the LBVH broad phase only");
    hipStream_t s = c.stream;
    const double* X0 = c.X[0].as<double>();
    const double* X1 = swept ? c.X[1].as<double>() : nullptr;
    c.cand_valid = false;
    c.n_ee = c.n_fv = c.n_vv = c.n_ev = 0;
    struct Tag { // stage names carry the query kind while this call runs
        Ctx& c;
        Tag(Ctx& c, bool swept) : c(c) { c.stage_tag = swept ? ".swept" : ".static"; }
        ~Tag() { c.stage_tag.clear(); }
    } tag(c, swept);
    if (c.nV == 0) {
        c.cand_valid = true;
        c.cand_swept = swept;
        return;
    }
    mesh_bounds(c, X0, X1, inflation);
    int axis = 0;
    if (sap) {
        // sweep axis: largest extent of the mesh box
        double* hb = static_cast<double*>(c.pinned);
        IPCG_HIP(hipMemcpyAsync(hb, c.aabb.p, sizeof(double) * 6, hipMemcpyDeviceToHost, s));
        IPCG_HIP(hipStreamSynchronize(s));
        for (int k = 1; k < 3; k++)
            if (hb[3 + k] - hb[k] > hb[3 + axis] - hb[axis]) axis = k;
        const TreeJob sets[3] = { { &c.tv, nullptr, 1, c.nV, false, nullptr, nullptr },
                                  { &c.te, c.E.as<int32_t>(), 2, c.nE, false, nullptr, nullptr },
                                  { &c.tf, c.F.as<int32_t>(), 3, c.nF, false, nullptr, nullptr } };
        sap_lists(c, sets, 3, X0, X1, inflation, axis);
    }
    c.row_order_valid = true; // c.aabb: the box of every scene
    const bool codim = c.n_cv > 0;
    {
        // vertex order (queries of the face tree), edge tree, face tree
        const bool fo = c.batched();
        TreeJob sets[TREES];
        int n = 0;
        if (!sap) {
            sets[n++] = { &c.tv, nullptr, 1, c.nV, false, nullptr, fo ? &c.h_voff : nullptr };
            sets[n++] = { &c.te, c.E.as<int32_t>(), 2, c.nE, true, nullptr,
                          fo ? &c.h_eoff : nullptr };
            sets[n++] = { &c.tf, c.F.as<int32_t>(), 3, c.nF, true, nullptr,
                          fo ? &c.h_foff : nullptr };
        }
        // codim lists (candidates.cpp:65-118): a tree over the codim vertices
        // (its own queries) and one over the codim edges; LBVH semantics with
        // either method
        if (codim) {
            sets[n++] = { &c.tcv, c.cv.as<int32_t>(), 1, c.n_cv, true, c.cv.as<int32_t>(),
                          fo ? &c.h_cvoff : nullptr };
            sets[n++] = { &c.tce, c.cev.as<int32_t>(), 2, c.n_ce, true, c.ce.as<int32_t>(),
                          fo ? &c.h_ceoff : nullptr };
        }
        build_trees(c, sets, n, X0, X1, inflation);
    }

    c.counters.reserve(sizeof(unsigned long long) * 4);
    Filter flt { c.E.as<int32_t>(), c.F.as<int32_t>(), c.has_patch ? c.patch.as<int32_t>() : nullptr,
                 c.n_dynamic, c.n_codim_filter };
    c.shard_cnt.reserve(4 * SHARD_CNT_BYTES + sizeof(WalkStatus));
    WalkStatus* const ws = reinterpret_cast<WalkStatus*>(c.shard_cnt.as<char>() + 4 * SHARD_CNT_BYTES);
    int* const status = &ws->status;
    unsigned* const claimed = &ws->claimed;
    c.shard_off.reserve(sizeof(int64_t) * 4 * (SHARDS + 1));
    unsigned long long* cnt[4];
    for (int k = 0; k < 4; k++) cnt[k] = c.shard_cnt.as<unsigned long long>() + k * SHARDS * SHARD_PAD;
    int64_t* scap[4] = { &c.scap_ee, &c.scap_fv, &c.scap_vv, &c.scap_ev };
    const int64_t guess[4] = { 16 * (int64_t)c.nE, 8 * (int64_t)c.nV, 4 * (int64_t)c.n_cv,
                               4 * (int64_t)c.n_cv };
    DevBuf* final_list[4] = { &c.cand_ee, &c.cand_fv, &c.cand_vv, &c.cand_ev };
    int64_t* final_n[4] = { &c.n_ee, &c.n_fv, &c.n_vv, &c.n_ev };
    const int lists = codim ? 4 : 2;
    const int qw = wave_queries((int64_t)c.nE + c.nV);
    const int64_t lanes = walk_lanes(c.nE, qw) + walk_lanes(c.nV, qw)
        + (codim ? 2 * walk_lanes(c.n_cv, qw) : 0);
    for (int attempt = 0; attempt < 3;) {
        const unsigned slots = reserve_slots(c, lanes);
        int* const deep = c.tr_deep.as<int>();
        // per-shard regions; their sum bounds a list until a retry grows it
        for (int k = 0; k < lists; k++) {
            if (*scap[k] == 0) *scap[k] = std::max<int64_t>(1024, guess[k] / SHARDS);
            c.cand_stage[k].reserve(sizeof(int2) * (size_t)(SHARDS * *scap[k]));
        }
        IPCG_HIP(hipMemsetAsync(c.shard_cnt.p, 0, 4 * SHARD_CNT_BYTES + sizeof(WalkStatus), s));
        const Shards S0 { cnt[0], c.scap_ee }, S1 { cnt[1], c.scap_fv };
        if (sap) {
            c.stage_begin("bp_sweep");
            if (c.nE >= 2)
                hipLaunchKernelGGL(k_sap_self, dim3(grid_for(c.nE, TR_BLOCK)), dim3(TR_BLOCK), 0, s,
                                   c.te.sbox.as<double>(), c.te.ids.as<uint32_t>(), c.nE, axis,
                                   flt, c.cand_stage[0].as<int2>(), S0);
            if (c.nF >= 1) {
                hipLaunchKernelGGL((k_sap_cross<true, false>), dim3(grid_for(c.nF, TR_BLOCK)),
                                   dim3(TR_BLOCK), 0, s, c.tf.sbox.as<double>(),
                                   c.tf.ids.as<uint32_t>(), c.nF, c.tv.sbox.as<double>(),
                                   c.tv.ids.as<uint32_t>(), c.nV, axis, flt,
                                   c.cand_stage[1].as<int2>(), S1);
                hipLaunchKernelGGL((k_sap_cross<false, true>), dim3(grid_for(c.nV, TR_BLOCK)),
                                   dim3(TR_BLOCK), 0, s, c.tv.sbox.as<double>(),
                                   c.tv.ids.as<uint32_t>(), c.nV, c.tf.sbox.as<double>(),
                                   c.tf.ids.as<uint32_t>(), c.nF, axis, flt,
                                   c.cand_stage[1].as<int2>(), S1);
            }
            c.stage_end();
        } else {
            const std::string tag = swept ? ".swept" : ".static";
            const TraverseArgs ee { c.te.box.as<float>(), c.te.ids.as<uint32_t>(), c.nE,
                                    c.te.nodes.as<Node>(), c.te.root.as<int32_t>(),
                                    c.te.leaf.as<int4>(), c.te.box.as<float>(), c.nE, flt,
                                    nullptr, c.cand_stage[0].as<int2>(), S0, deep, claimed,
                                    slots, status,
                                    forest_args(c, c.te), qw };
            const TraverseArgs fv { c.tv.box.as<float>(), c.tv.ids.as<uint32_t>(), c.nV,
                                    c.tf.nodes.as<Node>(), c.tf.root.as<int32_t>(),
                                    c.tf.leaf.as<int4>(), c.tf.box.as<float>(), c.nF, flt,
                                    nullptr, c.cand_stage[1].as<int2>(), S1, deep, claimed,
                                    slots, status,
                                    forest_args(c, c.tf), qw };
            if (c.nE >= 1 && c.nF >= 1) { // (a face brings its edges)
                c.stage_begin("bp_traverse_both");
                tuned_traverse(c, "bp_traverse_both" + tag, cnt[0], 2, claimed, [&](int b) {
                    if (swept) launch_both<1>(b, ee, fv, s);
                    else launch_both<0>(b, ee, fv, s);
                });
                c.stage_end();
            } else if (c.nE >= 2) {
                c.stage_begin("bp_traverse_ee");
                tuned_traverse(c, "bp_traverse_ee" + tag, cnt[0], 1, claimed, [&](int b) {
                    if (swept) launch_traverse<TR_EE, 1>(b, ee, s);
                    else launch_traverse<TR_EE, 0>(b, ee, s);
                });
                c.stage_end();
            }
        }
        if (codim) {
            c.stage_begin("bp_traverse_codim");
            const Shards S2 { cnt[2], c.scap_vv }, S3 { cnt[3], c.scap_ev };
            if (c.n_cv >= 2) {
                const TraverseArgs a { c.tcv.box.as<float>(), c.tcv.ids.as<uint32_t>(), c.n_cv,
                                       c.tcv.nodes.as<Node>(), c.tcv.root.as<int32_t>(),
                                       c.tcv.leaf.as<int4>(), c.tcv.box.as<float>(), c.n_cv, flt,
                                       c.cv.as<int32_t>(), c.cand_stage[2].as<int2>(), S2, deep,
                                       claimed, slots, status, forest_args(c, c.tcv), qw };
                if (swept) launch_traverse<TR_VV, 1>(TR_BLOCK, a, s);
                else launch_traverse<TR_VV, 0>(TR_BLOCK, a, s);
            }
            if (c.n_ce >= 1) {
                const TraverseArgs a { c.tcv.box.as<float>(), c.tcv.ids.as<uint32_t>(), c.n_cv,
                                       c.tce.nodes.as<Node>(), c.tce.root.as<int32_t>(),
                                       c.tce.leaf.as<int4>(), c.tce.box.as<float>(), c.n_ce, flt,
                                       c.cv.as<int32_t>(), c.cand_stage[3].as<int2>(), S3, deep,
                                       claimed, slots, status, forest_args(c, c.tce), qw };
                if (swept) launch_traverse<TR_EV, 1>(TR_BLOCK, a, s);
                else launch_traverse<TR_EV, 0>(TR_BLOCK, a, s);
            }
            c.stage_end();
        }
        IPCG_CHECK_LAUNCH();
        // the lists' counts and the walk status in one read-back
        ShardCounts kc[4];
        WalkStatus walk {};
        c.shard_sum.reserve(256);
        shard_counts_n(cnt[0], lists, c.shard_sum.as<unsigned long long>(),
                       c.shard_off.as<int64_t>(), c.pinned, s, kc, ws, &walk);
        const int st = walk.status;
        if (st & 2) throw Error(IPCG_ERR_NUMERIC, "LBVH build produced an invalid tree");
        if (st & 1) throw Error(IPCG_ERR_NUMERIC, "LBVH traversal stack overflow (depth > 64)");
        c.stat["bp.spill_stacks"] = walk.claimed;
        if (slots_short(c, st, slots, lanes)) continue;
        attempt++;
        bool again = false;
        for (int k = 0; k < lists; k++) {
            if (kc[k].max > *scap[k]) {
                *scap[k] = kc[k].max + kc[k].max / 4 + 1024;
                again = true;
            }
        }
        if (again) continue;
        c.stage_begin("bp_compact");
        for (int k = 0; k < 4; k++) {
            const int64_t m = k < lists ? kc[k].total : 0;
            final_list[k]->reserve(sizeof(int2) * (size_t)std::max<int64_t>(m, 1));
            if (m > 0)
                shard_compact(c.cand_stage[k].as<int2>(), *scap[k], kc[k].max,
                              final_list[k]->as<int2>(),
                              c.shard_off.as<int64_t>() + k * (SHARDS + 1), s);
            *final_n[k] = m;
        }
        c.stage_end();
        c.cand_valid = true;
        c.cand_swept = swept;
        return;
    }
    throw Error(IPCG_ERR_NUMERIC, "broad phase candidate lists kept outgrowing their regions");
}

// detect_edge_face_candidates (lbvh.cpp:771-784) over static boxes of
// positions slot 0: edge queries against a face LBVH, (edge, face) pairs
// into c.cand_ef.  The edge and face trees of an earlier broad phase are
// rebuilt here; its candidate lists stay valid.
void bp_edge_face(Ctx& c, double inflation)
{
    c.require_mesh();
    c.require_pos(0);
    c.n_ef = 0;
    if (c.nE == 0 || c.nF == 0) return;
    hipStream_t s = c.stream;
    const double* X0 = c.X[0].as<double>();
    struct Tag {
        Ctx& c;
        Tag(Ctx& c) : c(c) { c.stage_tag = ".ef"; }
        ~Tag() { c.stage_tag.clear(); }
    } tag(c);
    mesh_bounds(c, X0, nullptr, inflation);
    const bool fo = c.batched();
    const TreeJob sets[2] = {
        { &c.te, c.E.as<int32_t>(), 2, c.nE, false, nullptr, fo ? &c.h_eoff : nullptr },
        { &c.tf, c.F.as<int32_t>(), 3, c.nF, true, nullptr, fo ? &c.h_foff : nullptr }
    };
    build_trees(c, sets, 2, X0, nullptr, inflation);
    Filter flt { c.E.as<int32_t>(), c.F.as<int32_t>(), c.has_patch ? c.patch.as<int32_t>() : nullptr,
                 c.n_dynamic, c.n_codim_filter };
    c.counters.reserve(sizeof(unsigned long long) * 4);
    c.shard_cnt.reserve(4 * SHARD_CNT_BYTES + sizeof(WalkStatus));
    WalkStatus* const ws = reinterpret_cast<WalkStatus*>(c.shard_cnt.as<char>() + 4 * SHARD_CNT_BYTES);
    int* const status = &ws->status;
    unsigned* const claimed = &ws->claimed;
    c.shard_off.reserve(sizeof(int64_t) * 4 * (SHARDS + 1));
    unsigned long long* cnt = c.shard_cnt.as<unsigned long long>();
    const int qw = wave_queries(c.nE);
    const int64_t lanes = walk_lanes(c.nE, qw);
    for (int attempt = 0; attempt < 3;) {
        const unsigned slots = reserve_slots(c, lanes);
        if (c.scap_ef == 0) c.scap_ef = std::max<int64_t>(1024, 8 * (int64_t)c.nE / SHARDS);
        c.cand_stage[0].reserve(sizeof(int2) * (size_t)(SHARDS * c.scap_ef));
        IPCG_HIP(hipMemsetAsync(cnt, 0, SHARD_CNT_BYTES, s));
        IPCG_HIP(hipMemsetAsync(ws, 0, sizeof(WalkStatus), s));
        const Shards S0 { cnt, c.scap_ef };
        c.stage_begin("bp_traverse_ef");
        const TraverseArgs a { c.te.box.as<float>(), c.te.ids.as<uint32_t>(), c.nE,
                               c.tf.nodes.as<Node>(), c.tf.root.as<int32_t>(), c.tf.leaf.as<int4>(),
                               c.tf.box.as<float>(), c.nF, flt, nullptr, c.cand_stage[0].as<int2>(),
                               S0, c.tr_deep.as<int>(), claimed, slots, status,
                               forest_args(c, c.tf), qw };
        launch_traverse<TR_EF, 0>(TR_BLOCK, a, s);
        IPCG_CHECK_LAUNCH();
        c.stage_end();
        ShardCounts kc;
        WalkStatus walk {};
        c.shard_sum.reserve(256);
        shard_counts_n(cnt, 1, c.shard_sum.as<unsigned long long>(), c.shard_off.as<int64_t>(),
                       c.pinned, s, &kc, ws, &walk);
        const int st = walk.status;
        if (st & 2) throw Error(IPCG_ERR_NUMERIC, "LBVH build produced an invalid tree");
        if (st & 1) throw Error(IPCG_ERR_NUMERIC, "LBVH traversal stack overflow (depth > 64)");
        c.stat["bp.spill_stacks"] = walk.claimed;
        if (slots_short(c, st, slots, lanes)) continue;
        attempt++;
        if (kc.max > c.scap_ef) {
            c.scap_ef = kc.max + kc.max / 4 + 1024;
            continue;
        }
        c.cand_ef.reserve(sizeof(int2) * (size_t)std::max<int64_t>(kc.total, 1));
        if (kc.total > 0)
            shard_compact(c.cand_stage[0].as<int2>(), c.scap_ef, kc.max, c.cand_ef.as<int2>(),
                          c.shard_off.as<int64_t>(), s);
        c.n_ef = kc.total;
        return;
    }
    throw Error(IPCG_ERR_NUMERIC, "edge-face candidate list kept outgrowing its regions");
}

} // namespace ipcg
