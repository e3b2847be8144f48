// Signed point-to-mesh distance in FP64: nglod_mesh2sdf_f64
// (mesh2sdf.mesh2sdf_gpu, mesh2sdf_kernel.cu:307-616, 895-927).
//
// The distance is the minimum over the triangles, and a point is inside iff
// each of 13 lines through it meets a triangle on both sides.  Both need few
// of the triangles, so a call of more than a few pairs (pair_lanes) sorts the
// triangles along a Morton curve and builds a tree of boxes over them (8
// children per node, consecutive in that order).  Boxes are FP32 and wide
// enough for every rounding of the FP64 tests below them, so the triangles
// that are skipped could not have changed a result: the distance is the same
// minimum over the same FP64 values and the flags are the same flags as those
// of a loop over all triangles.
//
// 2^19 points (a third uniform in the box, the rest near the surface) and 5120
// triangles: 2.25 ms, of it 0.10 ms for the tree, 0.08 ms for the order of the
// points, 0.77 ms for the distances and 1.31 ms for the lines; 30.3 ms with
// every point against every triangle (FP64 issue, 2.7 G pairs).
#include "api_common.hpp"
#include "radix_sort.hpp"

namespace nglod {

__constant__ double kStab[13][3] = {
    {1.0f, 0.0f, 0.0f},
    {0.0f, 1.0f, 0.0f},
    {0.0f, 0.0f, 1.0f},
    {0.0f, 0.707106781f, 0.707106781f},
    {0.707106781f, 0.0f, 0.707106781f},
    {0.707106781f, 0.707106781f, 0.0f},
    {0.0f, 0.707106781f, -0.707106781f},
    {0.707106781f, 0.0f, -0.707106781f},
    {0.707106781f, -0.707106781f, 0.0f},
    {0.577350269f, 0.577350269f, 0.577350269f},
    {-0.577350269f, 0.577350269f, 0.577350269f},
    {0.577350269f, -0.577350269f, 0.577350269f},
    {0.577350269f, 0.577350269f, -0.577350269f},
};
constexpr int kDirs = 13;

// The 13 directions are axes, face diagonals and space diagonals, so a line
// is fixed by two or three of nine linear forms of its points, the same for
// all 13.  A line meets a box (or a triangle) only if those forms of the
// point lie in the box's intervals of them: nine interval tests per node
// serve all 13 lines.
enum : int { FX = 0, FY, FZ, FYmZ, FYpZ, FXmZ, FXpZ, FXmY, FXpY, kForms };
constexpr int kLineForms[kDirs][3] = {
    {FY, FZ, FZ},         {FX, FZ, FZ},         {FX, FY, FY},         {FX, FYmZ, FYmZ},     {FY, FXmZ, FXmZ},
    {FZ, FXmY, FXmY},     {FX, FYpZ, FYpZ},     {FY, FXpZ, FXpZ},     {FZ, FXpY, FXpY},     {FYmZ, FXmZ, FXmY},
    {FYmZ, FXpY, FXpZ},   {FXpY, FYpZ, FXmZ},   {FXmY, FXpZ, FYpZ},
};

__device__ __forceinline__ void point_forms(float x, float y, float z, float (&v)[kForms]) {
    v[FX] = x;
    v[FY] = y;
    v[FZ] = z;
    v[FYmZ] = y - z;
    v[FYpZ] = y + z;
    v[FXmZ] = x - z;
    v[FXpZ] = x + z;
    v[FXmY] = x - y;
    v[FXpY] = x + y;
}

// Per-triangle data of the distance: the vertices as given (their differences
// and products are formed again at each use: FP64 issue is idle there, the
// vector memory path is not) and the reciprocal squared lengths of the edges
// and of the normal.  degenerate: 1 if the normal is 0.
struct __align__(16) TriNear {
    float v[9];
    uint32_t degenerate;
    uint32_t pad[2];
    double i10, i21, i02, inor;
};

// Per-triangle data of the line tests.
struct __align__(16) TriLine {
    double a[3], v10[3], e2[3], pad;
    struct {
        double pvec[3];
        double idet;  // 0 where |det| < 1e-8 (no intersection)
    } dir[kDirs];
};

// The FP64 distance and stabbing arithmetic lets the compiler fuse a multiply
// and an add (one rounding instead of two): the library is otherwise built
// without contraction so that FP32 results follow the reference op by op, but
// here the bar is the distance to 1e-12 relative (1e-15 absolute) and exact
// signs, and the fused form issues about a quarter fewer FP64 instructions.
#define NGLOD_FP64_CONTRACT _Pragma("clang fp contract(fast)")

__device__ __forceinline__ double dot3(const double* a, const double* b) {
    NGLOD_FP64_CONTRACT
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
}
__device__ __forceinline__ void cross3(const double* a, const double* b, double* r) {
    NGLOD_FP64_CONTRACT
    r[0] = a[1] * b[2] - a[2] * b[1];
    r[1] = a[2] * b[0] - a[0] * b[2];
    r[2] = a[0] * b[1] - a[1] * b[0];
}

__device__ __forceinline__ double clamp01(double x) { return fmax(0.0, fmin(x, 1.0)); }
__device__ __forceinline__ double d2axmb(const double* a, double x, const double* b) {
    NGLOD_FP64_CONTRACT
    const double t0 = a[0] * x - b[0], t1 = a[1] * x - b[1], t2 = a[2] * x - b[2];
    return t0 * t0 + t1 * t1 + t2 * t2;
}

// The two records of a triangle (its nine floats), and its longest edge's square and
// 1 / its smallest determinant that is not taken for 0.
struct TriScale {
    double ee, worst;
};

__device__ __forceinline__ TriScale tri_records(const float* t, TriNear& N, TriLine& L) {
    NGLOD_FP64_CONTRACT
    double A[3], B[3], C[3], v10[3], v21[3], v02[3], nor[3];
    for (int k = 0; k < 3; ++k) {
        A[k] = t[k];
        B[k] = t[3 + k];
        C[k] = t[6 + k];
    }
    for (int k = 0; k < 3; ++k) {
        v10[k] = B[k] - A[k];
        v21[k] = C[k] - B[k];
        v02[k] = A[k] - C[k];
    }
    cross3(v10, v02, nor);
    for (int k = 0; k < 9; ++k) N.v[k] = t[k];
    N.i10 = 1.0 / dot3(v10, v10);
    N.i21 = 1.0 / dot3(v21, v21);
    N.i02 = 1.0 / dot3(v02, v02);
    N.inor = 1.0 / dot3(nor, nor);
    N.degenerate = (nor[0] == 0.0 && nor[1] == 0.0 && nor[2] == 0.0) ? 1u : 0u;
    for (int k = 0; k < 3; ++k) {
        L.a[k] = A[k];
        L.v10[k] = v10[k];
        L.e2[k] = -v02[k];
    }
    TriScale s;
    s.worst = 0.0;
    for (int i = 0; i < kDirs; ++i) {
        const double dir[3] = {kStab[i][0], kStab[i][1], kStab[i][2]};
        cross3(dir, L.e2, L.dir[i].pvec);
        const double det = dot3(v10, L.dir[i].pvec);
        L.dir[i].idet = (det > -1e-8 && det < 1e-8) ? 0.0 : 1.0 / det;
        s.worst = fmax(s.worst, fabs(L.dir[i].idet));
    }
    s.ee = fmax(dot3(v10, v10), fmax(dot3(v21, v21), dot3(v02, v02)));
    return s;
}

// ---------------------------------------------------------------------------
// The tree.  Level 0 is the sorted triangles, level l + 1 has one node per 8
// consecutive nodes of level l; the top level has at most 8 nodes.  Nodes are
// numbered in groups of 8 siblings, level by level.  A group is kept twice,
// as each walk reads it: per node its box and what lies below it (distance),
// and per linear form its nodes' intervals (lines).
constexpr int kMaxLevels = 10;
constexpr uint32_t kLeaf = 0x80000000u, kNone = 0xffffffffu;
constexpr int kBoundsBlocks = 64;

// below: the group of the node's children, kLeaf | triangle, or kNone past
// the level's last node.
struct __align__(16) Box {
    float lo[3];
    uint32_t below;
    float hi[3];
    uint32_t pad;
};

// Intervals as 16-bit steps over the mesh's range of each form: node k in half
// k / 4 of word k % 4.  The step of a value grows with it, so a value inside an
// interval has its step inside the interval's steps.  below: the children's
// group (or kLeaf | triangle) of node 0, each next node has the next.
struct __align__(16) Slabs {
    uint32_t lo[kForms][4], hi[kForms][4];
    uint32_t below, count, pad[2];
};
static_assert(sizeof(Slabs) % 16 == 0, "16-byte rows");

struct Tree {
    const TriNear* near;
    const TriLine* line;
    Box* boxes;                  // [groups][8]
    Slabs* slabs;                // [groups]
    int levels;                  // levels of nodes, the triangles' included
    uint32_t count[kMaxLevels];  // nodes of a level
    uint32_t goff[kMaxLevels];   // first group of a level
};

// Bounds of the finite vertices, one partial [6] per block (lo xyz, hi xyz).
__global__ __launch_bounds__(256) void mesh_bounds_kernel(const float* __restrict__ mesh, int64_t nf,
                                                          float* __restrict__ partial) {
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x; v < 3 * nf; v += (int64_t)gridDim.x * 256) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float p = mesh[3 * v + k];
            if (fabsf(p) < INFINITY) {
                lo[k] = fminf(lo[k], p);
                hi[k] = fmaxf(hi[k], p);
            }
        }
    }
    __shared__ float s[4][6];
#pragma unroll
    for (int k = 0; k < 3; ++k)
        for (int o = 32; o > 0; o >>= 1) {
            lo[k] = fminf(lo[k], __shfl_xor(lo[k], o));
            hi[k] = fmaxf(hi[k], __shfl_xor(hi[k], o));
        }
    if ((threadIdx.x & 63) == 0)
        for (int k = 0; k < 3; ++k) {
            s[threadIdx.x >> 6][k] = lo[k];
            s[threadIdx.x >> 6][3 + k] = hi[k];
        }
    __syncthreads();
    if (threadIdx.x < 6) {
        float v = s[0][threadIdx.x];
        for (int w = 1; w < 4; ++w) v = threadIdx.x < 3 ? fminf(v, s[w][threadIdx.x]) : fmaxf(v, s[w][threadIdx.x]);
        partial[6 * blockIdx.x + threadIdx.x] = v;
    }
}

// The bounds from the kBoundsBlocks partials, in every thread of a block of
// at least 64 threads (wave 0 reduces them).
struct Bounds {
    float lo[3], hi[3];
};

__device__ __forceinline__ Bounds load_bounds(const float* __restrict__ partial) {
    __shared__ float s[6];
    if (threadIdx.x < 64) {
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            float v = partial[6 * threadIdx.x + k];
            for (int o = 32; o > 0; o >>= 1) {
                const float w = __shfl_xor(v, o);
                v = k < 3 ? fminf(v, w) : fmaxf(v, w);
            }
            if (threadIdx.x == 0) s[k] = v;
        }
    }
    __syncthreads();
    Bounds b;
    for (int k = 0; k < 3; ++k) {
        b.lo[k] = s[k];
        b.hi[k] = s[3 + k];
    }
    return b;
}

// The 16-bit step of value v of form k: a monotone function of v.
__device__ __forceinline__ uint32_t form_step(const Bounds& b, int k, float v) {
    constexpr int axis[kForms][2] = {{0, 0}, {1, 1}, {2, 2}, {1, 2}, {1, 2}, {0, 2}, {0, 2}, {0, 1}, {0, 1}};
    const int i = axis[k][0], j = axis[k][1];
    float lo = b.lo[i], hi = b.hi[i];
    if (k >= 3) {
        const bool minus = (k & 1) != 0;
        lo += minus ? -b.hi[j] : b.lo[j];
        hi += minus ? -b.lo[j] : b.hi[j];
    }
    const float q = (v - lo) * (65535.0f / (hi - lo));
    return q > 0.0f ? (uint32_t)fminf(q, 65535.0f) : 0u;
}

// Spreads the low 10 bits of v to every third bit.
__device__ __forceinline__ uint32_t spread3(uint32_t v) {
    v &= 0x3FFu;
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

// Morton code of a point, `cells` cells per axis over the bounds (points
// outside them take the nearest cell; NaN cell 0).
__device__ __forceinline__ uint32_t morton_in(const Bounds& b, const float* p, float cells) {
    uint32_t key = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float q = (p[k] - b.lo[k]) / (b.hi[k] - b.lo[k]) * cells;
        key |= spread3(q > 0.0f ? (uint32_t)fminf(q, cells - 1.0f) : 0u) << k;
    }
    return key;
}

constexpr int kTriKeyBits = 30;    // 1024 cells per axis
constexpr int kPointKeyBits = 24;  // 256: finer cells do not make 64 points a tighter cluster

__global__ __launch_bounds__(256) void tri_keys_kernel(const float* __restrict__ mesh, uint32_t nf,
                                                       const float* __restrict__ partial,
                                                       uint32_t* __restrict__ keys) {
    const Bounds b = load_bounds(partial);
    const uint32_t f = blockIdx.x * 256 + threadIdx.x;
    if (f >= nf) return;
    const float* t = mesh + 9 * (size_t)f;
    float c[3];
    for (int k = 0; k < 3; ++k) c[k] = (t[k] + t[3 + k] + t[6 + k]) * (1.0f / 3.0f);
    keys[f] = morton_in(b, c, 1024.0f);
}

__global__ __launch_bounds__(256) void point_keys_kernel(const float* __restrict__ pts, uint32_t n,
                                                         const float* __restrict__ partial,
                                                         uint32_t* __restrict__ keys) {
    const Bounds b = load_bounds(partial);
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float p[3] = {pts[3 * (size_t)i], pts[3 * (size_t)i + 1], pts[3 * (size_t)i + 2]};
    keys[i] = morton_in(b, p, 256.0f);
}

// The FP64 record and the intervals of each triangle, in sorted order.
//
// Interval width.  The FP32 sums of a vertex or a point round by at most
// 2^-24 of |x| + |y|; the FP64 line test accepts a line that passes the
// triangle at a distance of up to 2 e |du| with |du| the error of its u and v:
// det and the numerators round by 6 * 2^-53 of R e and e^2 (R the distance
// from the point to the vertex, e the longest edge), so |du| <= 6.7e-16 (R e +
// e^2) / |det|, with the smallest |det| of the triangle's directions that is not taken
// for 0: that grows with the mesh's units as the triangle does (with 1e-8, the least
// it can be, it grew with their cube: an object 9000 units wide had nothing culled,
// 5120 triangles and 10^5 points 45.8 ms instead of 1.4).  A point outside the mesh's
// bounds has no hit on one side of an axis line, so R is at most their diagonal.  Both
// terms are taken several times over.  A triangle with a vertex that is not finite, or
// a determinant that is a good part rounding, gets unbounded intervals: it is
// looked at for every point.
__device__ __forceinline__ uint16_t* slab_half(uint32_t (&words)[4], uint32_t node) {
    return reinterpret_cast<uint16_t*>(&words[node & 3u]) + (node >> 2);
}

__global__ __launch_bounds__(128) void tri_prep_kernel(const float* __restrict__ mesh, uint32_t nf,
                                                       const uint32_t* __restrict__ order,
                                                       const float* __restrict__ partial, TriNear* __restrict__ near,
                                                       TriLine* __restrict__ line, Box* __restrict__ boxes,
                                                       Slabs* __restrict__ slabs) {
    NGLOD_FP64_CONTRACT
    const Bounds bd = load_bounds(partial);
    const uint32_t s = blockIdx.x * 128 + threadIdx.x;
    if (s >= (nf + 7) / 8 * 8) return;
    Box box;
    if (s >= nf) {
        for (int k = 0; k < 3; ++k) box.lo[k] = box.hi[k] = 0.0f;
        box.below = kNone;
        boxes[s] = box;
        return;
    }
    const float* t = mesh + 9 * (size_t)order[s];
    TriNear N;
    TriLine L;
    const TriScale sc = tri_records(t, N, L);
    near[s] = N;
    line[s] = L;
    float S = 0.0f, diag = 0.0f;
    for (int k = 0; k < 3; ++k) {
        S = fmaxf(S, fmaxf(fabsf(bd.lo[k]), fabsf(bd.hi[k])));
        diag += bd.hi[k] - bd.lo[k];
    }
    const float pad = 4e-6f * S + (float)(6e-15 * sc.worst * sc.ee * (sqrt(sc.ee) + (double)diag));
    float va[kForms], vb[kForms], vc[kForms];
    point_forms(t[0], t[1], t[2], va);
    point_forms(t[3], t[4], t[5], vb);
    point_forms(t[6], t[7], t[8], vc);
    bool finite = fabsf(pad) < INFINITY && 6.7e-16 * sc.worst * sc.ee < 0.25;
    for (int k = 0; k < 9; ++k) finite &= fabsf(t[k]) < INFINITY;
    Slabs& sl = slabs[s >> 3];
    for (int k = 0; k < kForms; ++k) {
        const float lo = fminf(va[k], fminf(vb[k], vc[k])) - pad, hi = fmaxf(va[k], fmaxf(vb[k], vc[k])) + pad;
        if (k < 3) {
            box.lo[k] = finite ? lo : -INFINITY;
            box.hi[k] = finite ? hi : INFINITY;
        }
        *slab_half(sl.lo[k], s & 7u) = finite ? (uint16_t)form_step(bd, k, lo) : (uint16_t)0;
        *slab_half(sl.hi[k], s & 7u) = finite ? (uint16_t)form_step(bd, k, hi) : (uint16_t)65535;
    }
    box.below = kLeaf | s;
    boxes[s] = box;
    if ((s & 7u) == 0) {
        sl.below = kLeaf | s;
        sl.count = min(8u, nf - s);
    }
}

// Node j of level l from its children, in items: 0..5 the box's bounds, then
// the slabs' steps, and last what lies below.
constexpr int kUpItems = 6 + 2 * kForms + 1;

__device__ __forceinline__ void up_one(const Tree& t, int l, uint32_t j, int q) {
    const uint32_t below = t.goff[l - 1] + j, group = t.goff[l] + (j >> 3);
    Box& box = t.boxes[(size_t)group * 8 + (j & 7u)];
    Slabs& sl = t.slabs[group];
    if (j >= t.count[l]) {
        if (q == kUpItems - 1) box.below = kNone;
        return;
    }
    const uint32_t cnt = min(8u, t.count[l - 1] - 8u * j);
    if (q < 6) {
        const Box* c = t.boxes + (size_t)below * 8;
        float v = q < 3 ? c[0].lo[q] : c[0].hi[q - 3];
        for (uint32_t k = 1; k < cnt; ++k) v = q < 3 ? fminf(v, c[k].lo[q]) : fmaxf(v, c[k].hi[q - 3]);
        (q < 3 ? box.lo[q] : box.hi[q - 3]) = v;
    } else if (q < kUpItems - 1) {
        const int f = (q - 6) >> 1;
        const bool upper = (q & 1) != 0;
        Slabs& c = t.slabs[below];
        uint16_t v = *slab_half(upper ? c.hi[f] : c.lo[f], 0);
        for (uint32_t k = 1; k < cnt; ++k) {
            const uint16_t w = *slab_half(upper ? c.hi[f] : c.lo[f], k);
            v = upper ? max(v, w) : min(v, w);
        }
        *slab_half(upper ? sl.hi[f] : sl.lo[f], j & 7u) = v;
    } else {
        box.below = below;
        if ((j & 7u) == 0) {
            sl.below = below;
            sl.count = min(8u, t.count[l] - j);
        }
    }
}

__device__ __forceinline__ uint32_t up_nodes(const Tree& t, int l) { return (t.count[l] + 7) / 8 * 8; }

__global__ __launch_bounds__(256) void tree_up_kernel(Tree t, int l) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    const uint64_t j = i / kUpItems;
    if (j < up_nodes(t, l)) up_one(t, l, (uint32_t)j, (int)(i % kUpItems));
}

// The small levels l0 .. top in one block.
__global__ __launch_bounds__(1024) void tree_top_kernel(Tree t, int l0) {
    for (int l = l0; l < t.levels; ++l) {
        for (uint32_t i = threadIdx.x; i < up_nodes(t, l) * kUpItems; i += 1024)
            up_one(t, l, i / kUpItems, (int)(i % kUpItems));
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Squared distance from p (p0 = p - the first vertex) to a triangle by the
// reference's edge/face rule, with the FP64 operations of a loop over the whole mesh.
// T: its vertices and reciprocals.
template <typename Tri>
__device__ __forceinline__ double edge_face_dist2(const Tri& T, const double* p0, const double* p, const double* v10,
                                                  const double* v21, const double* v02, const double* nor,
                                                  const double* c10, const double* c21, const double* c02) {
    NGLOD_FP64_CONTRACT
    const double p1[3] = {p[0] - T.v[3], p[1] - T.v[4], p[2] - T.v[5]};
    const double p2[3] = {p[0] - T.v[6], p[1] - T.v[7], p[2] - T.v[8]};
    const double s = copysign(1.0, dot3(c10, p0)) + copysign(1.0, dot3(c21, p1)) + copysign(1.0, dot3(c02, p2));
    double d2;
    if (s < 2.0) {
        const double e1 = d2axmb(v10, clamp01(dot3(v10, p0) * T.i10), p0);
        const double e2 = d2axmb(v21, clamp01(dot3(v21, p1) * T.i21), p1);
        const double e3 = d2axmb(v02, clamp01(dot3(v02, p2) * T.i02), p2);
        d2 = fmin(e1, fmin(e2, e3));
    } else {
        const double dn = dot3(nor, p0);
        d2 = dn * dn * T.inor;
    }
    return d2 < 0.0 ? 0.0 : d2;
}

// The distance for a triangle of the tree; INFINITY for a degenerate
// triangle, NaN where the arithmetic gives it (the minimum drops both).
__device__ __forceinline__ double tri_dist2(const TriNear& T, const double* p) {
    NGLOD_FP64_CONTRACT
    if (T.degenerate) return INFINITY;
    const double A[3] = {T.v[0], T.v[1], T.v[2]}, B[3] = {T.v[3], T.v[4], T.v[5]}, C[3] = {T.v[6], T.v[7], T.v[8]};
    const double v10[3] = {B[0] - A[0], B[1] - A[1], B[2] - A[2]};
    const double v21[3] = {C[0] - B[0], C[1] - B[1], C[2] - B[2]};
    const double v02[3] = {A[0] - C[0], A[1] - C[1], A[2] - C[2]};
    double nor[3], c10[3], c21[3], c02[3];
    cross3(v10, v02, nor);
    cross3(v10, nor, c10);
    cross3(v21, nor, c21);
    cross3(v02, nor, c02);
    const double p0[3] = {p[0] - A[0], p[1] - A[1], p[2] - A[2]};
    return edge_face_dist2(T, p0, p, v10, v21, v02, nor, c10, c21, c02);
}

// The bound a box must beat, from the best squared distance so far: FP32
// rounding up, with room for the rounding of the boxes' FP32 distances.
__device__ __forceinline__ float bound_of(double best) { return fmaxf((float)best * 1.00001f, 1e-37f); }

__device__ __forceinline__ float box_dist2(const Box& b, const float (&x)[3]) {
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float d = fmaxf(fmaxf(b.lo[k] - x[k], x[k] - b.hi[k]), 0.0f);
        s += d * d;
    }
    return s;
}

// Lane swaps within a row of 16 (DPP): xor 1, xor 2, mirror of 8, rotate by 8.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ double dpp_min(double v) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint64_t o = (uint64_t)dpp<CTRL>((uint32_t)b) | ((uint64_t)dpp<CTRL>((uint32_t)(b >> 32)) << 32);
    return fmin(v, __longlong_as_double((long long)o));
}
constexpr int kXor1 = 0xB1, kXor2 = 0x4E, kMirror8 = 0x141, kRotate8 = 0x128;

// Unsigned distances.  A wave takes 8 points (neighbours in space when
// ordered) and visits one group per step: lane 8 i + c holds point i against
// child c, so 64 box tests, and at a leaf up to 64 FP64 triangle distances,
// run at once.  The children some point needs go on the stack in LDS, the
// nearest on top; an entry that no point needs any more is dropped unvisited.
// The vector memory path bounds it: a node is two 16-byte loads and a triangle
// five (1.11 ms with a load per bound and the products of the edges stored,
// 0.77 ms so, 2^19 points and 5120 triangles).
//
// 64 points per wave against one child after another (wave-uniform, no
// divergence) took 4.1 ms instead: a few waves, those of points in the middle
// of the shape that are about as far from all its triangles, went through
// thousands of triangles in turn while the rest of the GPU had ended.
constexpr int kNearStack = 7 * kMaxLevels + 8;  // a step takes one entry and adds at most 8

__global__ __launch_bounds__(256) void mesh_near_kernel(const float* __restrict__ pts, int64_t first,
                                                        int64_t n, const uint32_t* __restrict__ order, Tree t,
                                                        float* __restrict__ dist, double* __restrict__ dist64) {
    __shared__ uint2 stacks[4][kNearStack];
    volatile uint2* stack = stacks[threadIdx.x >> 6];
    const uint32_t lane = lane_id(), c = lane & 7u;
    const int64_t s = first + ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * 8 + (lane >> 3);
    const bool valid = s < n;
    if (__ballot(valid) == 0) return;  // whole wave past the end (no barrier follows)
    const int64_t i = valid ? (order ? (int64_t)order[s] : s) : 0;
    float x[3] = {pts[3 * i], pts[3 * i + 1], pts[3 * i + 2]};
    const double p[3] = {x[0], x[1], x[2]};
    // a point that is not finite is culled by nothing: NaN has distance 0 from every box
    if (!(fabsf(x[0]) < INFINITY && fabsf(x[1]) < INFINITY && fabsf(x[2]) < INFINITY))
        x[0] = x[1] = x[2] = __builtin_nanf("");
    double best = INFINITY;
    float bound = valid ? INFINITY : -1.0f;
    uint32_t wbound = __float_as_uint(INFINITY);  // the largest bound of the wave's points
    uint32_t cur = t.goff[t.levels - 1];
    int sp = 0;
    for (;;) {
        const Box box = t.boxes[(size_t)cur * 8 + c];
        const float d2 = box_dist2(box, x);
        const bool pass = box.below != kNone && !(d2 > bound);
        const uint64_t m = __ballot(pass);
        if (__builtin_amdgcn_readfirstlane(box.below) & kLeaf) {  // node 0 of a group is never absent
            if (m != 0) {
                if (pass) best = fmin(best, tri_dist2(t.near[box.below & ~kLeaf], p));
                best = dpp_min<kMirror8>(dpp_min<kXor2>(dpp_min<kXor1>(best)));
                if (valid) bound = bound_of(best);
                wbound = 0u;
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    wbound = max(wbound, (uint32_t)max(__builtin_amdgcn_readlane((int)__float_as_uint(bound), 8 * k), 0));
            }
        } else {
            uint32_t mm = (uint32_t)m | (uint32_t)(m >> 32);
            mm |= mm >> 16;
            mm = (mm | (mm >> 8)) & 0xffu;
            // each child's distance to the nearest of the points that need it, the child in the low bits
            uint32_t key = pass ? ((__float_as_uint(d2) & ~7u) | c) : 0x7fffffffu;
            key = min(key, dpp<kRotate8>(key));
            const auto r16 = __builtin_amdgcn_permlane16_swap(key, key, false, false);
            key = min(r16[0], r16[1]);
            const auto r32 = __builtin_amdgcn_permlane32_swap(key, key, false, false);
            key = min(r32[0], r32[1]);
            int rank = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k)
                rank += ((mm >> k) & 1u) && (uint32_t)__builtin_amdgcn_readlane((int)key, k) > key ? 1 : 0;
            if (lane < 8 && ((mm >> lane) & 1u)) {
                stack[sp + rank].x = box.below;
                stack[sp + rank].y = key & ~7u;
            }
            sp += __popc(mm);
        }
        bool found = false;
        while (sp > 0 && !found) {
            --sp;
            cur = __builtin_amdgcn_readfirstlane(stack[sp].x);
            found = __builtin_amdgcn_readfirstlane(stack[sp].y) <= wbound;
        }
        if (!found) break;
    }
    if (valid && c == 0) {
        const double d = sqrt(best);
        dist[i] = (float)d;
        if (dist64) dist64[i] = d;
    }
}

// ---------------------------------------------------------------------------
typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u16x2_t as_u16x2(uint32_t w) { return __builtin_bit_cast(u16x2_t, w); }

// Signs: a point per lane.  A line is followed down the tree by its lane
// alone: on entry to a group the eight children are tested at once and the
// ones the line meets kept as a mask, so a lane's stack is one (group, mask)
// per level; at a leaf the FP64 test of each such triangle.  Ends once both
// sides have a hit.  Lanes of their own follow their lines' few nodes: a wave
// that walks its 64 points' 13 lines together enters the union of them.  The
// group loads bound it (vector memory path): 16-bit intervals halve them
// against FP32 ones (1.76 -> 1.31 ms at 2^19 points, 5120 triangles).
struct LineStack {
    uint32_t group[kMaxLevels][256];
    uint32_t mask[kMaxLevels][256];
};

template <int D>
__device__ __forceinline__ bool line_both_sides(const Tree& t, volatile LineStack* st, const double* p,
                                                const u16x2_t (&v)[kForms], bool all) {
    NGLOD_FP64_CONTRACT
    const int tid = threadIdx.x;
    bool ahead = false, behind = false;
    uint32_t cur = t.goff[t.levels - 1];
    int depth = 0;
    for (;;) {
        const Slabs& g = t.slabs[cur];
        const uint2 below = *reinterpret_cast<const uint2*>(&g.below);
        // bits of `out` that are set: where a form lies outside a node's interval
        u16x2_t out[4] = {};
#pragma unroll
        for (int f = 0; f < (kLineForms[D][1] == kLineForms[D][2] ? 2 : 3); ++f) {
            const int k = kLineForms[D][f];
            const uint4 l = *reinterpret_cast<const uint4*>(g.lo[k]), h = *reinterpret_cast<const uint4*>(g.hi[k]);
            const uint32_t lw[4] = {l.x, l.y, l.z, l.w}, hw[4] = {h.x, h.y, h.z, h.w};
#pragma unroll
            for (int w = 0; w < 4; ++w)
                out[w] |= (__builtin_elementwise_max(as_u16x2(lw[w]), v[k]) ^ v[k]) |
                          (__builtin_elementwise_min(as_u16x2(hw[w]), v[k]) ^ v[k]);
        }
        uint32_t mask = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const u16x2_t one = {1, 1};
            mask |= __builtin_bit_cast(uint32_t, __builtin_elementwise_min(out[w], one)) << w;
        }
        mask = (mask | (mask >> 12)) & 0xffu;  // nodes 0 .. 3 in the low halves, 4 .. 7 in the high
        mask = (all ? 0xffu : ~mask) & ((1u << below.y) - 1u);
        if (below.x & kLeaf) {
            while (mask != 0 && !(ahead && behind)) {
                const int c = __ffs((int)mask) - 1;
                mask &= mask - 1u;
                const TriLine& T = t.line[(below.x & ~kLeaf) + c];
                const double inv = T.dir[D].idet;
                if (inv == 0.0) continue;
                const double p0[3] = {p[0] - T.a[0], p[1] - T.a[1], p[2] - T.a[2]};
                double qvec[3];
                cross3(p0, T.v10, qvec);
                const double tnum = dot3(T.e2, qvec);
                const double u = dot3(p0, T.dir[D].pvec) * inv;
                if (u < 0.0 || u > 1.0) continue;
                const double dir[3] = {kStab[D][0], kStab[D][1], kStab[D][2]};
                const double w = dot3(dir, qvec) * inv;
                if (w < 0.0 || u + w > 1.0) continue;
                if (tnum * inv >= 0.0) ahead = true;
                else behind = true;
            }
            if (ahead && behind) return true;
        } else if (mask != 0) {
            st->group[depth][tid] = below.x;
            st->mask[depth][tid] = mask;
            ++depth;
        }
        if (depth == 0) return false;
        const uint32_t m = st->mask[depth - 1][tid];
        cur = st->group[depth - 1][tid] + (uint32_t)(__ffs((int)m) - 1);
        if ((m & (m - 1u)) == 0) --depth;
        else st->mask[depth - 1][tid] = m & (m - 1u);
    }
}

template <int D>
__device__ __forceinline__ bool lines_from(const Tree& t, volatile LineStack* st, const double* p,
                                           const u16x2_t (&v)[kForms], bool all) {
    if constexpr (D == kDirs)
        return true;
    else
        return line_both_sides<D>(t, st, p, v, all) && lines_from<D + 1>(t, st, p, v, all);
}

__global__ __launch_bounds__(256) void mesh_sign_kernel(const float* __restrict__ pts, int64_t n,
                                                        const uint32_t* __restrict__ order,
                                                        const float* __restrict__ partial, Tree t,
                                                        float* __restrict__ dist, double* __restrict__ dist64) {
    __shared__ LineStack st;
    const Bounds bd = load_bounds(partial);
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;  // no barrier follows
    const int64_t i = order ? (int64_t)order[s] : s;
    const float x[3] = {pts[3 * i], pts[3 * i + 1], pts[3 * i + 2]};
    const double p[3] = {x[0], x[1], x[2]};
    // a point that is not finite is looked at against every triangle
    const bool all = !(fabsf(x[0]) < INFINITY && fabsf(x[1]) < INFINITY && fabsf(x[2]) < INFINITY);
    // a point outside the mesh's bounds has no hit on one side of an axis
    const Box* top = t.boxes + (size_t)t.goff[t.levels - 1] * 8;
    bool in = true;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        float lo = top[0].lo[k], hi = top[0].hi[k];
        for (uint32_t c = 1; c < t.count[t.levels - 1]; ++c) {
            lo = fminf(lo, top[c].lo[k]);
            hi = fmaxf(hi, top[c].hi[k]);
        }
        in = in && !(x[k] < lo) && !(x[k] > hi);
    }
    if (!(in || all)) return;
    float f[kForms];
    point_forms(x[0], x[1], x[2], f);
    u16x2_t v[kForms];
#pragma unroll
    for (int k = 0; k < kForms; ++k) {
        const uint16_t q = (uint16_t)form_step(bd, k, f[k]);
        v[k] = u16x2_t{q, q};
    }
    if (lines_from<0>(t, &st, p, v, all)) {
        dist[i] = -dist[i];
        if (dist64) dist64[i] = -dist64[i];
    }
}

// ---------------------------------------------------------------------------
// Every point against every triangle, for few of either: no order, no tree, two
// launches.  `lanes` lanes of a wave take a point, each every lanes-th triangle of a
// tile in LDS; the minimum and the flags do not depend on the order.
//
// Bound: FP64 issue (11 ps a pair) where the points fill the GPU, else the chain of a
// lane's triangles (2.4 us each).  The tree's sorts and levels cost 100 us and more before
// its first triangle: 12 triangles and 10^4 points 158 us by the tree, 16 so.
struct PairTri {
    float v[9];
    uint32_t degenerate;
    double v10[3], v02[3], nor[3], c10[3], c21[3], c02[3], i10, i21, i02, inor;
    double pvec[kDirs][3], idet[kDirs];
};
constexpr int kPairTile = 64, kPairWords = sizeof(PairTri) / 8, kPairStride = kPairWords + 1;  // odd: over the banks
// the records take the place of the tree's
static_assert(8 * sizeof(PairTri) <= 8 * (sizeof(TriNear) + sizeof(TriLine) + sizeof(Box)) + sizeof(Slabs), "room");

__global__ __launch_bounds__(128) void pair_records_kernel(const float* __restrict__ mesh, uint32_t nf,
                                                           PairTri* __restrict__ out) {
    NGLOD_FP64_CONTRACT
    const uint32_t f = blockIdx.x * 128 + threadIdx.x;
    if (f >= nf) return;
    TriNear N;
    TriLine L;
    tri_records(mesh + 9 * (size_t)f, N, L);
    PairTri T;
    for (int k = 0; k < 9; ++k) T.v[k] = N.v[k];
    T.degenerate = N.degenerate;
    double v21[3];
    for (int k = 0; k < 3; ++k) {
        T.v10[k] = L.v10[k];
        v21[k] = (double)N.v[6 + k] - (double)N.v[3 + k];
        T.v02[k] = -L.e2[k];
    }
    cross3(T.v10, T.v02, T.nor);
    cross3(T.v10, T.nor, T.c10);
    cross3(v21, T.nor, T.c21);
    cross3(T.v02, T.nor, T.c02);
    T.i10 = N.i10;
    T.i21 = N.i21;
    T.i02 = N.i02;
    T.inor = N.inor;
    for (int d = 0; d < kDirs; ++d) {
        for (int k = 0; k < 3; ++k) T.pvec[d][k] = L.dir[d].pvec[k];
        T.idet[d] = L.dir[d].idet;
    }
    out[f] = T;
}

__global__ __launch_bounds__(256) void mesh_pairs_kernel(const float* __restrict__ pts, int64_t n, uint32_t nf,
                                                         uint32_t lanes, const PairTri* __restrict__ tris,
                                                         float* __restrict__ dist, double* __restrict__ dist64) {
    NGLOD_FP64_CONTRACT
    __shared__ double tile[kPairTile * kPairStride];
    const uint32_t q = threadIdx.x % lanes;
    const int64_t i = (int64_t)blockIdx.x * (256 / lanes) + threadIdx.x / lanes;
    const int64_t at = i < n ? i : n - 1;
    const double p[3] = {pts[3 * at], pts[3 * at + 1], pts[3 * at + 2]};
    double best = INFINITY;
    uint32_t flags = 0;
    for (uint32_t f0 = 0; f0 < nf; f0 += kPairTile) {
        const uint32_t cnt = min((uint32_t)kPairTile, nf - f0);
        const double* src = reinterpret_cast<const double*>(tris + f0);
        __syncthreads();
        for (uint32_t w = threadIdx.x; w < cnt * kPairWords; w += 256)
            tile[w / kPairWords * kPairStride + w % kPairWords] = src[w];
        __syncthreads();
        for (uint32_t k = q; k < cnt; k += lanes) {
            const PairTri& T = *reinterpret_cast<const PairTri*>(tile + k * kPairStride);
            const double p0[3] = {p[0] - T.v[0], p[1] - T.v[1], p[2] - T.v[2]};
            const double v21[3] = {(double)T.v[6] - T.v[3], (double)T.v[7] - T.v[4], (double)T.v[8] - T.v[5]};
            if (!T.degenerate)
                best = fmin(best, edge_face_dist2(T, p0, p, T.v10, v21, T.v02, T.nor, T.c10, T.c21, T.c02));
            double qvec[3];
            cross3(p0, T.v10, qvec);
            const double e2[3] = {-T.v02[0], -T.v02[1], -T.v02[2]};
            const double tnum = dot3(e2, qvec);
#pragma unroll
            for (int d = 0; d < kDirs; ++d) {
                const double inv = T.idet[d];
                if (inv == 0.0) continue;
                const double u = dot3(p0, T.pvec[d]) * inv;
                if (u < 0.0 || u > 1.0) continue;
                const double dir[3] = {kStab[d][0], kStab[d][1], kStab[d][2]};
                const double w = dot3(dir, qvec) * inv;
                if (w < 0.0 || u + w > 1.0) continue;
                flags |= tnum * inv >= 0.0 ? 1u << d : 1u << (kDirs + d);
            }
        }
    }
    for (uint32_t o = lanes / 2; o > 0; o >>= 1) {
        best = fmin(best, __shfl_xor(best, (int)o));
        flags |= (uint32_t)__shfl_xor((int)flags, (int)o);
    }
    if (i >= n || q != 0) return;
    const double d = flags == (1u << 2 * kDirs) - 1u ? -sqrt(best) : sqrt(best);
    dist[i] = (float)d;
    if (dist64) dist64[i] = d;
}

// ---------------------------------------------------------------------------
static size_t up256(size_t b) { return (b + 255) / 256 * 256; }

struct SdfLayout {
    Tree tree;
    size_t near, line, boxes, slabs, bounds, sort, total;
    size_t psort, ordered_total;
};

// n = 0: without the point order.
static void sdf_layout(int64_t n, int64_t nf, SdfLayout* L) {
    memset(L, 0, sizeof(*L));
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t at = off;
        off += up256(bytes);
        return at;
    };
    uint64_t c = (uint64_t)nf, groups = 0;
    int l = 0;
    for (;; ++l) {
        L->tree.count[l] = (uint32_t)c;
        L->tree.goff[l] = (uint32_t)groups;
        groups += (c + 7) / 8;
        if (c <= 8) break;
        c = (c + 7) / 8;
    }
    L->tree.levels = l + 1;
    L->near = take((size_t)nf * sizeof(TriNear));
    L->line = take((size_t)nf * sizeof(TriLine));
    L->boxes = take((size_t)groups * 8 * sizeof(Box));
    L->slabs = take((size_t)groups * sizeof(Slabs));
    L->bounds = take(kBoundsBlocks * 6 * sizeof(float));
    L->sort = take(sort_workspace_bytes(nf));
    L->total = off + 8;  // the caller's workspace is 8-byte aligned, the tables 16
    if (n > 0) L->psort = take(sort_workspace_bytes(n));
    L->ordered_total = off + 8;
}

// Triangles and points are numbered with 32 bits here (2^30 triangles would
// need 700 GB of workspace), the count that kMaxLevels levels hold.
constexpr int64_t kMaxFaces = (int64_t)1 << 30;
constexpr int64_t kMaxOrdered = (int64_t)1 << 31;

// Lanes per point for every point against every triangle; 0: the tree.  Icospheres and a
// cube, us, tree / pairs: 12 triangles 110 / 13 with 1000 points, 274 / 72 with 2^19, 687 /
// 247 with 2^21; 20 triangles 687 / 475; 80 triangles 240 / 22 with 1000, 342 / 273 with
// 2^18, 485 / 513 with 2^19; 320 triangles 414 / 61 with 1000, 411 / 229 with 16000, 407 / 399
// with 64000; 1280 triangles 681 / 214 with 1000, 730 / 459 with 4000, 700 / 858 with 16000 (5120:
// 1286 / 821 and 1218 / 1795 with 1000 and 4000, and one point 400 / 814).  Lanes, 80 triangles: 4000
// points 41 with 64, 63 with 4, 190 with 1; 16000 130, 64, 190; 64000 467, 111, 192; 2^18
// 1848, 399, 273: beyond 4 the lanes' different triangles are bank conflicts.
static uint32_t pair_lanes(int64_t n, int64_t nf) {
    if (n <= 4096 ? nf > 1280 : nf > 24 && (nf > 320 || n * nf > (int64_t)1 << 24)) return 0;
    return n <= 4096 ? 64 : n <= 1 << 16 ? 4 : n <= 1 << 17 ? 2 : 1;
}

}  // namespace nglod

using namespace nglod;

extern "C" {

size_t nglod_mesh2sdf_workspace_size(int64_t nf) {
    if (nf <= 0 || nf > kMaxFaces) return 0;
    SdfLayout L;
    sdf_layout(0, nf, &L);
    return L.total;
}

size_t nglod_mesh2sdf_ordered_workspace_size(int64_t n, int64_t nf) {
    if (nf <= 0 || nf > kMaxFaces) return 0;
    SdfLayout L;
    sdf_layout(n > 0 && n <= kMaxOrdered ? n : 0, nf, &L);
    return L.ordered_total;
}

int nglod_mesh2sdf_f64(const float* points, int64_t n, const float* mesh, int64_t nf, float* dist, double* dist64,
                       void* workspace, size_t workspace_bytes, void* stream) {
    if (n < 0 || nf < 0) return fail(NGLOD_ERR_ARG, "negative size");
    if (n == 0) return NGLOD_OK;
    if (nf == 0) return fail(NGLOD_ERR_ARG, "mesh has no triangles");
    if (!points || !mesh || !dist) return fail(NGLOD_ERR_ARG, "NULL pointer");
    if (nf > kMaxFaces) return fail(NGLOD_ERR_WORKSPACE, "workspace too small or misaligned");
    SdfLayout L;
    sdf_layout(n <= kMaxOrdered ? n : 0, nf, &L);
    if (!workspace || workspace_bytes < L.total || ((uintptr_t)workspace & 7))
        return fail(NGLOD_ERR_WORKSPACE, "workspace too small or misaligned");
    // a workspace with room for the points' order has them visited in it
    const bool ordered = n <= kMaxOrdered && workspace_bytes >= L.ordered_total;
    hipStream_t s = (hipStream_t)stream;
    char* w = (char*)(((uintptr_t)workspace + 15) & ~(uintptr_t)15);
    Tree& t = L.tree;
    t.near = (const TriNear*)(w + L.near);
    t.line = (const TriLine*)(w + L.line);
    t.boxes = (Box*)(w + L.boxes);
    t.slabs = (Slabs*)(w + L.slabs);
    float* bounds = (float*)(w + L.bounds);
    const uint32_t nt = (uint32_t)nf;
    if (const uint32_t lanes = pair_lanes(n, nf)) {
        hipLaunchKernelGGL(pair_records_kernel, dim3((nt + 127) / 128), dim3(128), 0, s, mesh, nt, (PairTri*)w);
        const int64_t per = 256 / lanes;
        hipLaunchKernelGGL(mesh_pairs_kernel, dim3((unsigned)((n + per - 1) / per)), dim3(256), 0, s, points, n, nt,
                           lanes, (const PairTri*)w, dist, dist64);
        return check_launch("mesh_pairs_kernel");
    }
    const SortBuffers ts = sort_buffers(w + L.sort, nf);
    hipLaunchKernelGGL(mesh_bounds_kernel, dim3(kBoundsBlocks), dim3(256), 0, s, mesh, nf, bounds);
    hipLaunchKernelGGL(tri_keys_kernel, dim3((nt + 255) / 256), dim3(256), 0, s, mesh, nt, bounds, ts.keys[0]);
    const int tb = launch_sort(ts, nf, kTriKeyBits, s);
    hipLaunchKernelGGL(tri_prep_kernel, dim3((nt + 7 + 127) / 128), dim3(128), 0, s, mesh, nt, ts.vals[tb], bounds,
                       (TriNear*)(w + L.near), (TriLine*)(w + L.line), t.boxes, t.slabs);
    int l = 1;
    for (; l < t.levels && t.count[l] > 512; ++l)
        hipLaunchKernelGGL(tree_up_kernel, dim3((unsigned)((((uint64_t)t.count[l] + 7) * kUpItems + 255) / 256)),
                           dim3(256), 0, s, t, l);
    if (l < t.levels) hipLaunchKernelGGL(tree_top_kernel, dim3(1), dim3(1024), 0, s, t, l);
    int rc = check_launch("tree_top_kernel");
    if (rc) return rc;
    const uint32_t* order = nullptr;
    if (ordered) {
        const SortBuffers ps = sort_buffers(w + L.psort, n);
        hipLaunchKernelGGL(point_keys_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, points, (uint32_t)n,
                           bounds, ps.keys[0]);
        order = ps.vals[launch_sort(ps, n, kPointKeyBits, s)];
        rc = check_launch("sort_scatter_kernel");
        if (rc) return rc;
    }
    constexpr int64_t kSlice = (int64_t)1 << 28;  // 8 threads per point: below the 2^32 threads of a launch
    for (int64_t f = 0; f < n; f += kSlice)
        hipLaunchKernelGGL(mesh_near_kernel, dim3((unsigned)(((n - f < kSlice ? n - f : kSlice) + 31) / 32)), dim3(256),
                           0, s, points, f, n, order, t, dist, dist64);
    hipLaunchKernelGGL(mesh_sign_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, points, n, order, bounds,
                       t, dist, dist64);
    return check_launch("mesh_sign_kernel");
}

}  // extern "C"
