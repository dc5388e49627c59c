// Spatial-hash broadphase and vertex-face CCD for gfx950.
//
// Broadphase build (SpatialHashSystem, SpatialHashSystem.cpp:88-121, 276-413):
//   triangle centroid -> cell coordinates -> key (dense grid index or -1
//   outside, or a hashed table slot) -> stable radix sort of (key, id) ->
//   cell ranges [start, end].
// Candidates: an unsorted table of the faces by cell, built with one atomic
//   per entry; each vertex (edge) visits the cells around it once, so that
//   every distinct pair comes up exactly once and no list of pairs is sorted
//   or stored to be de-duplicated.
// Narrowphase: ExtendedVFTest (CCD.cpp:1733-1808) per candidate whose swept
//   boxes meet, FP64 only in the coplanarity cubic / time-of-impact solve
//   (CCD.cpp:48-113).
// Response: VFResolveTest/VFResolveNew (CCD.cpp:1996-2090) evaluated for all
//   contacts against the same positions, fixes summed per vertex in 2^-32 m
//   fixed point (integer sums are order independent, so the result does not
//   depend on atomic ordering) and applied as the mean fix per vertex.
// Paths are relative to PositionBasedDynamicsCUDA/PositionBasedDynamicsCUDA/.
#include <algorithm>
#include <climits>
#include <mutex>
#include <type_traits>

#include "pbd_internal.hpp"
#include "pbd_math.hpp"

namespace pbd {

// ---------------------------------------------------------------------------
// device scan (exclusive, int64 totals kept in int)
// ---------------------------------------------------------------------------
constexpr int SB = 1024;  // elements per scan block (256 threads x 4)

__global__ __launch_bounds__(256) void k_scan_blocks(const int* __restrict__ in, int* __restrict__ out, int n,
                                                     int* __restrict__ sums) {
    __shared__ int s[256];
    int base = blockIdx.x * SB, t = threadIdx.x;
    int v[4], tot = 0;
    for (int k = 0; k < 4; k++) {
        int i = base + t * 4 + k;
        v[k] = i < n ? in[i] : 0;
        tot += v[k];
    }
    s[t] = tot;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        int a = t >= off ? s[t - off] : 0;
        __syncthreads();
        s[t] += a;
        __syncthreads();
    }
    int run = s[t] - tot;
    for (int k = 0; k < 4; k++) {
        int i = base + t * 4 + k;
        if (i < n) out[i] = run;
        run += v[k];
    }
    if (t == 255) sums[blockIdx.x] = s[255];
}

__global__ __launch_bounds__(256) void k_scan_add(int* __restrict__ out, int n, const int* __restrict__ sums) {
    int i = blockIdx.x * SB + threadIdx.x;
    int add = sums[blockIdx.x];
    for (int k = 0; k < 4; k++, i += 256)
        if (i < n) out[i] += add;
}

__global__ __launch_bounds__(1024) void k_scan_single(int* __restrict__ a, int n) {
    __shared__ int part[1024];
    int t = threadIdx.x;
    int per = (n + 1023) / 1024;
    int b = t * per, e = min(n, b + per);
    int s = 0;
    for (int i = b; i < e; i++) s += a[i];
    part[t] = s;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        int v = t >= off ? part[t - off] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    int run = part[t] - s;
    for (int i = b; i < e; i++) {
        int v = a[i];
        a[i] = run;
        run += v;
    }
}

void device_scan(hipStream_t s, const int* in, int* out, int n, int* tmp) {
    if (n <= 0) return;
    int nb = (n + SB - 1) / SB;
    hipLaunchKernelGGL(k_scan_blocks, dim3(nb), dim3(256), 0, s, in, out, n, tmp);
    hipLaunchKernelGGL(k_scan_single, dim3(1), dim3(1024), 0, s, tmp, nb);
    hipLaunchKernelGGL(k_scan_add, dim3(nb), dim3(256), 0, s, out, n, tmp);
    PBD_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// broadphase
// ---------------------------------------------------------------------------
__device__ __forceinline__ int cell_key(const HashCfg& g, int x, int y, int z) {
    if (g.mode == 0) {
        if (x < 0 || y < 0 || z < 0 || x >= g.size[0] || y >= g.size[1] || z >= g.size[2]) return -1;
        return (int)(((unsigned)z * (unsigned)g.size[1]) * (unsigned)g.size[0] + (unsigned)y * (unsigned)g.size[0] +
                     (unsigned)x);
    }
    unsigned h = ((unsigned)x * 73856093u) ^ ((unsigned)y * 19349663u) ^ ((unsigned)z * 83492791u);
    return (int)(h & ((1u << g.table_bits) - 1u));
}

// A vertex position from the library's float4 records or from 3 floats per
// vertex (the C ABI's layout).
__device__ __forceinline__ float4 vload(const float4* __restrict__ p, int i) { return p[i]; }
__device__ __forceinline__ float4 vload(const float* __restrict__ p, int i) {
    return make_float4(p[3 * (size_t)i], p[3 * (size_t)i + 1], p[3 * (size_t)i + 2], 0.0f);
}

// centroid (a+b+c)/3 per component (evalTriCentroids) and its cell
// (calcGridPosCPU: floor((c - start)/cell)).
template <typename P>
__device__ __forceinline__ void tri_cell(const HashCfg& g, const P* __restrict__ p, const int* __restrict__ tris,
                                         int t, int* gp) {
    float4 a = vload(p, tris[3 * t]), b = vload(p, tris[3 * t + 1]), c = vload(p, tris[3 * t + 2]);
    float cx = (a.x + b.x + c.x) / 3, cy = (a.y + b.y + c.y) / 3, cz = (a.z + b.z + c.z) / 3;
    gp[0] = (int)floorf((cx - g.start[0]) / g.cell[0]);
    gp[1] = (int)floorf((cy - g.start[1]) / g.cell[1]);
    gp[2] = (int)floorf((cz - g.start[2]) / g.cell[2]);
}

// Keys of the triangles, one workgroup per sort tile, which also counts the
// first digit; the workgroups behind the tiles set the cell ranges to -1.
// Keys are stored plus 1, so that -1 (outside the grid) sorts first, as in the
// reference's signed sort.  BOUNDED: a triangle with a vertex index outside
// [0, nv) is given key -1 instead of being read.
constexpr int KEY_THREADS = 1024, FILL_INTS = 16384;

template <bool BOUNDED, typename P>
__global__ __launch_bounds__(KEY_THREADS) void k_tri_keys(HashCfg g, const P* __restrict__ p, int nv,
                                                          const int* __restrict__ tris, int nt, int ntiles,
                                                          uint32_t* __restrict__ keys1, int* __restrict__ raw,
                                                          int* __restrict__ counts, int* __restrict__ cstart,
                                                          int* __restrict__ cend, int quads) {
    const int tid = threadIdx.x;
    if ((int)blockIdx.x >= ntiles) {
        const int per = (g.ncells + FILL_INTS - 1) / FILL_INTS, f = blockIdx.x - ntiles;
        int* a = f < per ? cstart : cend;
        const long long from = (long long)(f < per ? f : f - per) * FILL_INTS;
        const int n = (int)min((long long)FILL_INTS, g.ncells - from);
        a += from;
        int i = 0;
        if (quads) {  // both arrays are 16-byte aligned
            for (int j = tid; j < n / 4; j += KEY_THREADS) reinterpret_cast<int4*>(a)[j] = make_int4(-1, -1, -1, -1);
            i = n & ~3;
        }
        for (i += tid; i < n; i += KEY_THREADS) a[i] = -1;
        return;
    }
    __shared__ int h[256];
    if (tid < 256) h[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RADIX_TILE / KEY_THREADS; r++) {
        const int t = blockIdx.x * RADIX_TILE + r * KEY_THREADS + tid;
        if (t >= nt) break;
        int k = -1;
        bool read = true;
        if (BOUNDED) {
            const int a = tris[3 * t], b = tris[3 * t + 1], c = tris[3 * t + 2];
            read = a >= 0 && a < nv && b >= 0 && b < nv && c >= 0 && c < nv;
        }
        if (read) {
            int gp[3];
            tri_cell(g, p, tris, t, gp);
            k = cell_key(g, gp[0], gp[1], gp[2]);
        }
        keys1[t] = (uint32_t)(k + 1);
        raw[t] = k;
        atomicAdd(&h[(k + 1) & 255], 1);
    }
    __syncthreads();
    if (tid < 256) counts[blockIdx.x * 256 + tid] = h[tid];
}

// Correct ranges of each key in the sorted array (the reference's
// findCellStartCPU misses some starts, SpatialHashSystem.cpp:357-387).
__global__ __launch_bounds__(256) void k_cell_ranges(const int* __restrict__ keys, int n, int* __restrict__ cstart,
                                                     int* __restrict__ cend) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int k = keys[i];
    if (k < 0) return;
    if (i == 0 || keys[i - 1] != k) cstart[k] = i;
    if (i == n - 1 || keys[i + 1] != k) cend[k] = i;
}

// The sorted table: keys (signed) and triangle ids in key order, unsorted
// keys, cell ranges.  tk / tv: room for nt, hist: radix_hist_ints(nt).
// Launches: keys with the first digit's counts and the ranges' fill, two per
// digit less one, the ranges (522,000 triangles, 2^22 cells: 128 us before,
// 53 us so).
template <bool BOUNDED, typename P>
static void build_sorted(hipStream_t s, const HashCfg& g, const P* p, int nv, const int* tris, int nt, uint32_t* ok,
                         uint32_t* ov, int* raw, int* cstart, int* cend, uint32_t* tk, uint32_t* tv, int* hist) {
    int bits = 1;
    while (bits < 32 && ((1ll << bits) < (long long)g.ncells + 1)) bits++;
    uint32_t* src = radix_passes(bits) % 2 ? tk : ok;
    const int tiles = radix_tiles(nt);
    const long long fill = 2ll * ((g.ncells + (long long)FILL_INTS - 1) / FILL_INTS);
    const int quads = ((uintptr_t)cstart | (uintptr_t)cend) % 16 == 0;
    if (tiles + fill > 0)
        hipLaunchKernelGGL((k_tri_keys<BOUNDED, P>), dim3((unsigned)(tiles + fill)), dim3(KEY_THREADS), 0, s, g, p, nv, tris,
                           nt, tiles, src, raw, hist, cstart, cend, quads);
    radix_sort(s, src, nullptr, tk, tv, ok, ov, nt, bits, hist, true, 1u);
    if (nt > 0)
        hipLaunchKernelGGL(k_cell_ranges, dim3((nt + 255) / 256), dim3(256), 0, s, (const int*)ok, nt, cstart, cend);
    PBD_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Candidate pairs.
//
// Centroid cells (FindNeighbors over every triangle as CCD_SH_Extended
// consumes it, SpatialHashSystem.cpp:134-187, CCD.cpp:1541-1586): (v, f) with
// v a vertex of some triangle t whose cell is valid, f in the 27 cells around
// t's cell, v not in f.  Edge pairs likewise from the cells of two triangles.
//
// Swept boxes (a conservative alternative, since the centroid cells miss faces
// larger than a cell): v is a vertex of some triangle, v not in f, and v's box
// over the substep, AABB(x_v, p_v), meets f's box over the substep, AABB of the
// six points x_f*, p_f*, widened per side by 4 thickness plus 1e-6 |bound|.
// The narrowphase accepts a vertex within 2 thickness of the face plane and
// inside the face's barycentric band of width thickness / mean edge, i.e.
// within sqrt(13) thickness of the face, at an interpolated position inside
// both boxes, so every pair it accepts is a candidate: the contact set equals
// that of the all-pairs test (CCD_N2, CCD.cpp:1040-1098).
//
// Faces go into a hash table by cell: slot counts (one atomic per entry, whose
// return value is the entry's place in its slot), slot offsets (one scan
// pass), the entries.  A group of 32 lanes takes a vertex (an edge): its lanes
// look up one cell each, then share the cells' entries evenly.  Each cell is
// visited once per vertex, so a pair comes up once.  The form this replaces
// made the pairs of every triangle (3.7 times as many on a folded 256 x 256
// cloth), stored them, sorted them twice and compacted them: 2.6 ms per
// detection there against 0.15 ms for the table, the visit and the narrowphase.
// ---------------------------------------------------------------------------
constexpr int SWEPT_MAX_CELLS = 4096;  // cells of the caller's grid one box may span
constexpr int ENTRY_MAX_CELLS = 64;    // cells of one level of the table's grid a face is entered in (any at the last)

__device__ __forceinline__ float widen_lo(float v, float m) { return v - (m + 1e-6f * fabsf(v)); }
__device__ __forceinline__ float widen_hi(float v, float m) { return v + (m + 1e-6f * fabsf(v)); }

// The cell of v along axis k, of cells `scale` times as long.
__device__ __forceinline__ int cell_coord(const HashCfg& g, float v, int k, float scale = 1.0f) {
    float c = floorf((v - g.start[k]) / (g.cell[k] * scale));
    c = fminf(fmaxf(c, -536870912.0f), 536870912.0f);  // keeps hi - lo + 1 within int
    int i = (int)c;
    if (g.mode == 0) i = min(max(i, 0), g.size[k] - 1);  // clamping keeps overlapping ranges overlapping
    return i;
}

struct SweptBox {
    float lo[3], hi[3];
};

__device__ __forceinline__ void box_add(SweptBox& b, float4 a) {
    const float c[3] = {a.x, a.y, a.z};
    for (int k = 0; k < 3; k++) {
        b.lo[k] = fminf(b.lo[k], c[k]);
        b.hi[k] = fmaxf(b.hi[k], c[k]);
    }
}

__device__ __forceinline__ SweptBox vertex_box(const float4 X, const float4 P) {
    SweptBox b;
    b.lo[0] = fminf(X.x, P.x); b.hi[0] = fmaxf(X.x, P.x);
    b.lo[1] = fminf(X.y, P.y); b.hi[1] = fmaxf(X.y, P.y);
    b.lo[2] = fminf(X.z, P.z); b.hi[2] = fmaxf(X.z, P.z);
    return b;
}

// Slot of a cell in the table (any hash does: entries carry their cell).
__device__ __forceinline__ unsigned cell_slot(int x, int y, int z, unsigned mask) {
    unsigned h = ((unsigned)x * 73856093u) ^ ((unsigned)y * 19349663u) ^ ((unsigned)z * 83492791u);
    h ^= h >> 15;
    return h & mask;
}

// A face as the visits read it, half a cache line: its widened swept box, its
// vertices, whether the box may rule pairs out (face_cullable), and its cell.
// Centroid-cell tables hold the records themselves (one entry per face), so
// that a visit reads a slot's faces side by side and nothing else of them.
struct alignas(64) FaceRec {
    float lo[3];
    int v0;
    float hi[3];
    int v1;
    int v2, cull, face;
    int cx, cy, cz;
    int pad[2];
};

// Whether a vertex outside the face's swept box widened by 4.5 thickness cannot
// pass the narrowphase's floating-point tests: the face keeps a good shape
// over the whole step (doubled area at least 0.05 of its longest edge squared,
// bounded below from the start's area and the edges' changes), so barycentric
// coordinates carry a relative error of about 1e-4, and the thickness is not
// tiny beside the edges, so the widening covers that error with room to spare.
// Pairs with other faces always go to the narrowphase.
__device__ __forceinline__ bool face_cullable(const float4* X, const float4* P, float th) {
    const V3 e1 = mk(X[1].x - X[0].x, X[1].y - X[0].y, X[1].z - X[0].z);
    const V3 e2 = mk(X[2].x - X[0].x, X[2].y - X[0].y, X[2].z - X[0].z);
    const V3 d1 = mk(P[1].x - P[0].x - e1.x, P[1].y - P[0].y - e1.y, P[1].z - P[0].z - e1.z);
    const V3 d2 = mk(P[2].x - P[0].x - e2.x, P[2].y - P[0].y - e2.y, P[2].z - P[0].z - e2.z);
    const V3 c = cross(e1, e2);
    const float l1 = sqrtf(dot(e1, e1)), l2 = sqrtf(dot(e2, e2)), m1 = sqrtf(dot(d1, d1)), m2 = sqrtf(dot(d2, d2));
    const V3 e3 = sub(e2, e1);
    const float longest = fmaxf(fmaxf(l1, l2), sqrtf(dot(e3, e3))) + m1 + m2;
    const float area = sqrtf(dot(c, c)) - (l1 * m2 + l2 * m1 + m1 * m2);
    return area >= 0.05f * (longest * longest) && th >= 4e-3f * longest;  // false for NaN
}

// Half-spaces that hold every vertex that can touch a face (cullable faces;
// others: all of space).  The narrowphase accepts a vertex at a time t whose
// distance from the face's plane is at most 2 thickness and whose barycentric
// coordinates are at least -e, e = thickness / mean edge length.  Along a
// direction m such a point lies below the extended corners
// (1 + 3 e) m.c_k - e sum(m.c), which are linear in t, plus 2 thickness
// |m.n(t)|.  m are the outward normals of the edges in the face's plane at
// t = 1/2, for which |m.n(t)| is bounded by the change of the edges, and the
// plane's normal, both ways.  The slack covers the rounding of the
// narrowphase's coordinates (relative to their size) and of its barycentric
// coordinates (1e-4 for cullable faces).  Coordinates are relative to a corner.
struct FaceAxes {
    float4 edge[3];  // m, highest m.c
    float4 plane;    // n, highest n.c
    float4 origin;   // the corner, lowest n.c
};

__device__ __forceinline__ FaceAxes face_axes(const float4* X, const float4* P, float th) {
    V3 c[2][3];
    float size = 0.0f;
    for (int k = 0; k < 3; k++) {
        c[0][k] = mk(X[k].x - X[0].x, X[k].y - X[0].y, X[k].z - X[0].z);
        c[1][k] = mk(P[k].x - X[0].x, P[k].y - X[0].y, P[k].z - X[0].z);
        size = fmaxf(size, fmaxf(fmaxf(fabsf(X[k].x), fabsf(X[k].y)), fabsf(X[k].z)));
        size = fmaxf(size, fmaxf(fmaxf(fabsf(P[k].x), fabsf(P[k].y)), fabsf(P[k].z)));
    }
    const V3 e1 = c[0][1], e2 = c[0][2], e3 = sub(e2, e1);
    const V3 d1 = sub(sub(c[1][1], c[1][0]), e1), d2 = sub(sub(c[1][2], c[1][0]), e2), d3 = sub(d2, d1);
    auto len = [](V3 a) { return sqrtf(dot(a, a)); };
    const float l1 = len(e1), l2 = len(e2), l3 = len(e3), m1 = len(d1), m2 = len(d2), m3 = len(d3);
    const float area = len(cross(e1, e2)) - (l1 * m2 + l2 * m1 + m1 * m2);  // lowest over the step
    const float mean = (l1 + l2 + l3 - (m1 + m2 + m3)) / 3.0f;
    const float e = 1.001f * th / mean;
    const float turn = fminf(1.0f, 1e-3f + (0.5f * (l1 * m2 + l2 * m1) + 0.75f * m1 * m2) / area);
    const float slack = 0.5f * th + 4e-6f * size;
    FaceAxes r;
    r.origin = make_float4(X[0].x, X[0].y, X[0].z, -INFINITY);
    r.plane = r.edge[0] = r.edge[1] = r.edge[2] = make_float4(0.0f, 0.0f, 0.0f, INFINITY);
    if (!(mean >= 0.25f * fmaxf(fmaxf(l1, l2), l3)) || !face_cullable(X, P, th)) return r;
    V3 h[3];
    for (int k = 0; k < 3; k++) h[k] = scale(0.5f, mk(c[0][k].x + c[1][k].x, c[0][k].y + c[1][k].y, c[0][k].z + c[1][k].z));
    const V3 big = cross(sub(h[1], h[0]), sub(h[2], h[0]));
    const V3 n = scale(1.0f / len(big), big);
    auto range = [&](V3 m, float* lo, float* hi) {
        *lo = INFINITY;
        *hi = -INFINITY;
        for (int t = 0; t < 2; t++) {
            const float a = dot(m, c[t][0]), b = dot(m, c[t][1]), d = dot(m, c[t][2]), s = e * (a + b + d);
            *hi = fmaxf(*hi, fmaxf(fmaxf(a, b), d) * (1.0f + 3.0f * e) - s);
            *lo = fminf(*lo, fminf(fminf(a, b), d) * (1.0f + 3.0f * e) - s);
        }
    };
    float lo, hi;
    for (int k = 0; k < 3; k++) {
        const V3 along = sub(h[k == 2 ? 0 : k + 1], h[k]), o = cross(along, n);
        const V3 m = scale(1.0f / len(o), o);
        range(m, &lo, &hi);
        r.edge[k] = make_float4(m.x, m.y, m.z, hi + 2.0f * th * turn + slack);
    }
    range(n, &lo, &hi);
    r.plane = make_float4(n.x, n.y, n.z, hi + 2.0f * th + slack);
    r.origin.w = lo - 2.0f * th - slack;
    return r;
}

// Whether the vertex stays outside one of the half-spaces (false for NaN).
__device__ __forceinline__ bool axes_miss(const FaceAxes& f, float4 x, float4 p) {
    const V3 a = mk(x.x - f.origin.x, x.y - f.origin.y, x.z - f.origin.z);
    const V3 b = mk(p.x - f.origin.x, p.y - f.origin.y, p.z - f.origin.z);
    // the rounding of the vertex's own coordinates along its way
    const float own = 2e-6f * fmaxf(fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fabsf(x.z)),
                                    fmaxf(fmaxf(fabsf(p.x), fabsf(p.y)), fabsf(p.z)));
    bool out = false;
    for (int k = 0; k < 3; k++) {
        const V3 m = mk(f.edge[k].x, f.edge[k].y, f.edge[k].z);
        out = out || fminf(dot(m, a), dot(m, b)) - own > f.edge[k].w;
    }
    const V3 n = mk(f.plane.x, f.plane.y, f.plane.z);
    const float na = dot(n, a), nb = dot(n, b);
    return out || fminf(na, nb) - own > f.plane.w || fmaxf(na, nb) + own < f.origin.w;
}

__device__ __forceinline__ FaceRec face_record(int f, const float4* __restrict__ x, const float4* __restrict__ p,
                                               const int* __restrict__ tris, float th, float margin) {
    FaceRec r;
    r.face = f;
    r.cx = r.cy = r.cz = 0;
    r.pad[0] = r.pad[1] = 0;
    r.v0 = tris[3 * f];
    r.v1 = tris[3 * f + 1];
    r.v2 = tris[3 * f + 2];
    const float4 X[3] = {x[r.v0], x[r.v1], x[r.v2]}, P[3] = {p[r.v0], p[r.v1], p[r.v2]};
    SweptBox b = vertex_box(X[0], X[0]);
    for (int k = 1; k < 3; k++) box_add(b, X[k]);
    for (int k = 0; k < 3; k++) box_add(b, P[k]);
    for (int k = 0; k < 3; k++) {
        r.lo[k] = widen_lo(b.lo[k], margin);
        r.hi[k] = widen_hi(b.hi[k], margin);
    }
    r.cull = face_cullable(X, P, th) ? 1 : 0;
    return r;
}

__device__ __forceinline__ bool box_misses(const SweptBox& b, const FaceRec& r) {
    return b.lo[0] > r.hi[0] || r.lo[0] > b.hi[0] || b.lo[1] > r.hi[1] || r.lo[1] > b.hi[1] || b.lo[2] > r.hi[2] ||
           r.lo[2] > b.hi[2];
}

// Centroid cells: the face's cell and place in its slot.  tcell[t] = (cell,
// slot), slot -1 outside a dense grid.
__global__ __launch_bounds__(256) void k_face_cells(HashCfg g, const float4* __restrict__ p,
                                                    const int* __restrict__ tris, int nt, unsigned mask,
                                                    int* __restrict__ cnt, int4* __restrict__ tcell,
                                                    int* __restrict__ rank) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nt) return;
    int gp[3];
    tri_cell(g, p, tris, t, gp);
    const bool in = cell_key(g, gp[0], gp[1], gp[2]) >= 0;
    const unsigned slot = cell_slot(gp[0], gp[1], gp[2], mask);
    tcell[t] = make_int4(gp[0], gp[1], gp[2], in ? (int)slot : -1);
    rank[t] = in ? atomicAdd(&cnt[slot], 1) : 0;
}

__global__ __launch_bounds__(256) void k_cell_fill(int nt, const int4* __restrict__ tcell, const int* __restrict__ rank,
                                                   const int* __restrict__ cnt, const int* __restrict__ end,
                                                   const float4* __restrict__ x, const float4* __restrict__ p,
                                                   const int* __restrict__ tris, float th, FaceRec* __restrict__ ent,
                                                   FaceAxes* __restrict__ axes) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nt) return;
    const int4 c = tcell[t];
    if (c.w < 0) return;
    if (axes) {
        const int3 v = make_int3(tris[3 * t], tris[3 * t + 1], tris[3 * t + 2]);
        const float4 X[3] = {x[v.x], x[v.y], x[v.z]}, P[3] = {p[v.x], p[v.y], p[v.z]};
        axes[t] = face_axes(X, P, th);
    }
    FaceRec r = face_record(t, x, p, tris, th, 4.5f * th);
    r.cx = c.x;
    r.cy = c.y;
    r.cz = c.z;
    ent[end[c.w] - cnt[c.w] + rank[t]] = r;
}

// Each slot's place among the entries: end[slot] (END) or its start.  Order
// among workgroups is whatever their atomics make it: few workgroups, since
// these are served one after the other (2^19 slots: 26 us with one per 256
// slots).
constexpr int PLACE_SLOTS = 4096;
template <bool END>
__global__ __launch_bounds__(256) void k_slot_places(const int4* __restrict__ cnt, int nslots, int4* __restrict__ place,
                                                     unsigned long long* __restrict__ total) {
    constexpr int Q = PLACE_SLOTS / 1024;
    __shared__ int wave[4], base;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int i0 = blockIdx.x * (PLACE_SLOTS / 4) + wv * (Q * 64) + lane;  // in quads of slots
    int4 c[Q];
    int before[Q], run = 0;
    for (int k = 0; k < Q; k++) {
        c[k] = 4 * (i0 + 64 * k) < nslots ? cnt[i0 + 64 * k] : make_int4(0, 0, 0, 0);
        int sum = c[k].x + c[k].y + c[k].z + c[k].w;
        const int mine = sum;
        for (int off = 1; off < 64; off <<= 1) {
            const int o = __shfl_up(sum, off);
            if (lane >= off) sum += o;
        }
        before[k] = run + sum - mine;
        run += __shfl(sum, 63);
    }
    if (lane == 0) wave[wv] = run;
    __syncthreads();
    if (threadIdx.x == 0) base = (int)atomicAdd(total, (unsigned long long)(wave[0] + wave[1] + wave[2] + wave[3]));
    __syncthreads();
    int at = base;
    for (int w = 0; w < wv; w++) at += wave[w];
    for (int k = 0; k < Q; k++) {
        if (4 * (i0 + 64 * k) >= nslots) break;
        int4 r;
        r.x = at + before[k] + (END ? c[k].x : 0);
        r.y = r.x + (END ? c[k].y : c[k].x);
        r.z = r.y + (END ? c[k].z : c[k].y);
        r.w = r.z + (END ? c[k].w : c[k].z);
        place[i0 + 64 * k] = r;
    }
}

// Swept boxes: face records (their margin defines the candidate set), the
// cells of the table's own grid they cover counted per slot.  The grid has
// SWEPT_LEVELS levels, each of cells SWEPT_FACTOR times as long as those of the
// one below: a face goes to the lowest where it covers at most ENTRY_MAX_CELLS
// cells, and vertices look in every level that holds faces.  So neither faces
// of very different size nor a motion over many cells make entries or visits
// many (a folded 512 x 512 cloth moving 8 edges along each axis: 27 ms a
// detection, 571 ms when faces over 64 cells went to a list that every vertex
// tested).  The narrowphase's half-spaces are made here, where the corners are
// loaded anyway (571,000 faces: 185 us without them, 193 with).
__device__ __forceinline__ unsigned level_slot(int x, int y, int z, int level, unsigned mask) {
    return (cell_slot(x, y, z, 0xffffffffu) + (unsigned)level * 0x9E3779B1u) & mask;
}

__global__ __launch_bounds__(256) void k_swept_faces(HashCfg g, HashCfg gi, const float4* __restrict__ x,
                                                     const float4* __restrict__ p, const int* __restrict__ tris, int nt,
                                                     float th, unsigned mask, int* __restrict__ cnt,
                                                     int4* __restrict__ fcell, FaceRec* __restrict__ rec,
                                                     FaceAxes* __restrict__ axes, DetectCounts* __restrict__ c) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nt) return;
    const FaceRec r = face_record(f, x, p, tris, th, 4.0f * th);
    const float4 X[3] = {x[r.v0], x[r.v1], x[r.v2]}, P[3] = {p[r.v0], p[r.v1], p[r.v2]};
    axes[f] = face_axes(X, P, th);
    long long span = 1;
    // per-axis bounds first: the product of three spans of up to 2^31 overflows
    for (int k = 0; k < 3; k++)
        span *= (long long)min(cell_coord(g, r.hi[k], k) - cell_coord(g, r.lo[k], k) + 1, SWEPT_MAX_CELLS + 1);
    rec[f] = r;
    const bool over = span > SWEPT_MAX_CELLS;  // the detection is refused
    if (over) c->face_span = 1;
    int lo[3], hi[3], level = 0;
    for (float scale = 1.0f;; level++, scale *= (float)SWEPT_FACTOR) {
        int n = 1;
        for (int k = 0; k < 3; k++) {
            lo[k] = cell_coord(gi, r.lo[k], k, scale);
            hi[k] = over ? lo[k] : cell_coord(gi, r.hi[k], k, scale);
            n *= min(hi[k] - lo[k] + 1, ENTRY_MAX_CELLS + 1);
        }
        if (n <= ENTRY_MAX_CELLS || level == SWEPT_LEVELS - 1) break;
    }
    fcell[2 * f] = make_int4(lo[0], lo[1], lo[2], level);
    fcell[2 * f + 1] = make_int4(hi[0], hi[1], hi[2], 0);
    c->level[level] = 1;
    for (int z = lo[2]; z <= hi[2]; z++)
        for (int y = lo[1]; y <= hi[1]; y++)
            for (int xx = lo[0]; xx <= hi[0]; xx++) atomicAdd(&cnt[level_slot(xx, y, z, level, mask)], 1);
}

// The cell of an entry, 9 bits per axis (a face covers fewer than CODE_SPAN
// cells along each, so it cannot cover two that agree in them), per axis whether
// it is the face's lowest cell, and the level.
constexpr int CODE_SPAN = 512;
__device__ __forceinline__ int cell_code(int x, int y, int z) { return (x & 511) | ((y & 511) << 9) | ((z & 511) << 18); }

// place: each slot's start, moved up by every entry stored; it ends at the
// slot's end.  FACE_LANES lanes share a face's cells, since every entry waits
// for its atomic (128 x 128 drape, 118,000 to 198,000 entries: 17.4 us with a
// thread per face, 14.4 so; counting waits for none and gains nothing by it).
// Places past 2^31 compare as unsigned: such a detection is refused, and until
// then nothing may be stored out of range.
constexpr int FACE_LANES = 8;
__global__ __launch_bounds__(256) void k_swept_fill(int nt, const int4* __restrict__ fcell, unsigned mask,
                                                    int* __restrict__ place, int2* __restrict__ ent, unsigned cap) {
    const int f = (blockIdx.x * blockDim.x + threadIdx.x) / FACE_LANES, lane = threadIdx.x % FACE_LANES;
    if (f >= nt) return;
    const int4 lo = fcell[2 * f], hi = fcell[2 * f + 1];
    const int wx = hi.x - lo.x + 1, wy = hi.y - lo.y + 1, n = wx * wy * (hi.z - lo.z + 1);
    for (int i = lane; i < n; i += FACE_LANES) {
        const int z = i / (wx * wy), j = i - z * (wx * wy), y = j / wx, xx = j - y * wx;
        const unsigned at = (unsigned)atomicAdd(&place[level_slot(lo.x + xx, lo.y + y, lo.z + z, lo.w, mask)], 1);
        const unsigned first = (xx == 0 ? 1u << 27 : 0) | (y == 0 ? 1u << 28 : 0) | (z == 0 ? 1u << 29 : 0);
        if (at < cap)
            ent[at] = make_int2(f, (int)((unsigned)cell_code(lo.x + xx, lo.y + y, lo.z + z) | first | (unsigned)lo.w << 30));
    }
}
static_assert(SWEPT_LEVELS <= 4, "two bits of an entry hold the level");

// Pairs a wave has found, appended in runs to the global list.  Atomics on one
// address are served one after the other, about 13 ns each here, so one length
// for the whole list bounded every visit (26,000 runs on the folded 256 x 256
// cloth: 340 of 371 us).  The list is NEAR_BUCKETS lists of `cap` pairs, each
// with its length in a line of its own; a wave goes on to another one after
// every run, so that the lists fill evenly whatever wave finds the most.
constexpr int VISIT_WAVES = 4, VISIT_BUF = 256;
struct PairSink {
    int2* buf;       // this wave's LDS
    int n;           // wave-uniform
    int bucket;      // wave-uniform
    DetectCounts* c;
    int2* out;
    unsigned cap;    // per bucket
    __device__ __forceinline__ void flush() {
        const int lane = threadIdx.x & 63;
        unsigned at = 0;
        if (lane == 0) at = atomicAdd(&c->bucket[bucket].near, (unsigned)n);
        at = __shfl(at, 0);
        int2* o = out + (size_t)bucket * cap;
        for (int i = lane; i < n; i += 64)
            if (at + i < cap) o[at + i] = buf[i];
        n = 0;
        bucket = (bucket + 17) % NEAR_BUCKETS;
    }
    __device__ __forceinline__ void count(int pairs) {
        for (int off = 32; off > 0; off >>= 1) pairs += __shfl_xor(pairs, off);
        if ((threadIdx.x & 63) == 0 && pairs) atomicAdd(&c->bucket[bucket].pairs, (unsigned long long)pairs);
    }
    // Called by all lanes of the wave.
    __device__ __forceinline__ void add(bool hit, int a, int b) {
        const unsigned long long m = __ballot(hit);
        if (!m) return;
        const int lane = threadIdx.x & 63;
        if (hit) buf[n + __popcll(m & ((1ull << lane) - 1ull))] = make_int2(a, b);
        n += __popcll(m);
        if (n > VISIT_BUF - 64) flush();
    }
};

// Data parallel primitives over the 32 lanes of a group.
template <int CTRL>
__device__ __forceinline__ int dpp(int v, int old) {
    return __builtin_amdgcn_update_dpp(old, v, CTRL, 0xf, 0xf, false);
}
template <class Op>
__device__ __forceinline__ int group_reduce(int v, Op&& op) {
    v = op(v, dpp<0xb1>(v, v));   // lanes xor 1
    v = op(v, dpp<0x4e>(v, v));   // lanes xor 2
    v = op(v, dpp<0x141>(v, v));  // half rows mirrored: the other four of eight
    v = op(v, dpp<0x140>(v, v));  // rows mirrored: the other eight of sixteen
    return op(v, __builtin_amdgcn_ds_swizzle(v, 0x401f));  // lanes xor 16
}
// Sum of the lanes up to and including this one.
__device__ __forceinline__ int group_scan(int v) {
    v += dpp<0x111>(v, 0);  // one lane up the row, then 2, 4, 8
    v += dpp<0x112>(v, 0);
    v += dpp<0x114>(v, 0);
    v += dpp<0x118>(v, 0);
    // the last lane of rows 0 and 2 to all of rows 1 and 3
    return v + __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
}
__device__ __forceinline__ void lds_ready() {  // this wave's LDS writes, to its own lanes
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// LDS of a group of 32 lanes.
constexpr int BOX_CELLS = 256, RUN_WINDOW = 1024;
struct GroupLds {
    unsigned cover[BOX_CELLS / 32];     // the cells of a box that are visited
    unsigned starts[RUN_WINDOW / 32];   // entries of the window that start a run
    int4 run[64];                       // cell, and where its entries lie less those of the runs before
};

// One round of a group's visit: every lane brings two cells q with n entries
// from `start` on (0: none); calls f(e, cell) for every entry, the lanes taking
// them in turn, and f(-1, cell) for the lanes left over.  An entry finds its
// run by counting the starts before it: a bit per entry in LDS, and one LDS
// read of the run (a binary search by shuffles took 14 LDS operations an
// entry; with it the visit of the folded 256 x 256 cloth took 119 us, 105 so).
// Both groups of a wave stay in the loops until the longer is done, so f may
// use wave-wide operations.
template <class F>
__device__ __forceinline__ void visit_runs(GroupLds& lds, const int3* q, const int* start, const int* n, F&& f) {
    const int lane = threadIdx.x & 63, l = lane & 31;
    const int sum = group_scan(n[0] + n[1]);
    const int total = __shfl(sum, 31, 32);
    const int before[2] = {sum - n[0] - n[1], sum - n[1]};
    const unsigned below = (1u << l) - 1u;
    unsigned has[2];
    for (int c = 0; c < 2; c++) {
        const unsigned long long m = __ballot(n[c] > 0);
        has[c] = lane < 32 ? (unsigned)m : (unsigned)(m >> 32);
    }
    int id = __popc(has[0] & below) + __popc(has[1] & below);
    __builtin_amdgcn_wave_barrier();  // the round before is done with the lists
    for (int c = 0; c < 2; c++)
        if (n[c] > 0) lds.run[id++] = make_int4(q[c].x, q[c].y, q[c].z, start[c] - before[c]);
    const int longest = max(total, __shfl_xor(total, 32));
    int runs = 0;  // that start before the current entries
    for (int w0 = 0; w0 < longest; w0 += RUN_WINDOW) {
        __builtin_amdgcn_wave_barrier();
        lds.starts[l] = 0;
        lds_ready();
        for (int c = 0; c < 2; c++) {
            const int at = before[c] - w0;
            if (n[c] > 0 && at >= 0 && at < RUN_WINDOW) atomicOr(&lds.starts[at >> 5], 1u << (at & 31));
        }
        lds_ready();
        const int w1 = min(longest, w0 + RUN_WINDOW);
        for (int b = w0; b < w1; b += 32) {
            const unsigned word = lds.starts[(b - w0) >> 5];
            const int i = b + l;
            const int4 r = lds.run[i < total ? runs + __popc(word & (0xffffffffu >> (31 - l))) - 1 : 0];
            runs += __popc(word);
            f(i < total ? i + r.w : -1, make_int3(r.x, r.y, r.z));
        }
    }
}
static_assert(RUN_WINDOW == 32 * 32, "a lane clears one word of the window");

// What a hub's unit visits (see HubRounds).
struct HubItem {
    const int* set;
    int unit, place;
};

// Whether c is a valid cell and (x, y, z) is within one cell of it.
__device__ __forceinline__ bool near_cell(int4 c, int x, int y, int z) {
    return c.w >= 0 && abs(c.x - x) <= 1 && abs(c.y - y) <= 1 && abs(c.z - z) <= 1;
}
// Cell l (0..26) of the 27 around c.
__device__ __forceinline__ int3 around(int4 c, int l) {
    return make_int3(c.x + l % 3 - 1, c.y + l / 3 % 3 - 1, c.z + l / 9 - 1);
}

// The entries of a lane's two cells q of round r of `cells`; whether there are any.
template <class Cells>
__device__ __forceinline__ bool cell_runs(const Cells& cells, const HashCfg& g, int r, const int* __restrict__ cnt,
                                          const int* __restrict__ end, unsigned mask, int3* q, int* start, int* n) {
    for (int c = 0; c < 2; c++) {
        const bool mine = cells.cell(g, r, c, &q[c]);
        const unsigned slot = mine ? cell_slot(q[c].x, q[c].y, q[c].z, mask) : 0u;
        const int k = cnt[slot], e = end[slot];
        n[c] = mine ? k : 0;
        start[c] = e - k;
    }
    return n[0] + n[1] > 0;
}

// The cells around a group's own triangles (up to HUB_FACES), each once, two
// per lane and round (most boxes have 27 to 64 cells, which then take one round
// of memory latencies): the cells of the box of their cells that lie around one
// of them.  A box of more than BOX_CELLS cells takes the 27 cells around one
// triangle after the other instead, without those that lie around an earlier one.
constexpr int HUB_FACES = 32;
struct CellRounds {
    const GroupLds* lds;
    const int* list;
    const int4* tcell;
    int deg, rounds;
    bool boxed;
    int3 lo, w;
    // Called by all lanes of the wave.
    __device__ __forceinline__ void start(GroupLds& g, const int* list_, int deg_, const int4* tcell_, const HubItem&) {
        lds = &g;
        list = list_;
        tcell = tcell_;
        deg = deg_;
        const int l = threadIdx.x & 31;
        const int4 c = l < deg ? tcell[list[l]] : make_int4(0, 0, 0, -1);
        const bool valid = c.w >= 0;
        auto least = [](int a, int b) { return min(a, b); };
        auto most = [](int a, int b) { return max(a, b); };
        lo = make_int3(group_reduce(valid ? c.x : INT_MAX, least), group_reduce(valid ? c.y : INT_MAX, least),
                       group_reduce(valid ? c.z : INT_MAX, least));
        const int3 hi = make_int3(group_reduce(valid ? c.x : INT_MIN, most), group_reduce(valid ? c.y : INT_MIN, most),
                                  group_reduce(valid ? c.z : INT_MIN, most));
        long long n = 0;
        w = make_int3(1, 1, 1);
        if (hi.x >= lo.x) {
            const long long top = BOX_CELLS + 1;
            w = make_int3((int)min((long long)hi.x - lo.x + 3, top), (int)min((long long)hi.y - lo.y + 3, top),
                          (int)min((long long)hi.z - lo.z + 3, top));
            n = (long long)w.x * w.y * w.z;
        }
        lo = make_int3(lo.x - 1, lo.y - 1, lo.z - 1);
        boxed = n <= BOX_CELLS;
        rounds = boxed ? ((int)n + 63) / 64 : deg;
        // mark the 27 cells around each triangle
        __builtin_amdgcn_wave_barrier();  // the group before is done with `cover`
        if (l < BOX_CELLS / 32) g.cover[l] = 0;
        lds_ready();
        const int at = valid ? ((c.z - lo.z) * w.y + c.y - lo.y) * w.x + c.x - lo.x : -1;
        const int off = ((l / 9 - 1) * w.y + l / 3 % 3 - 1) * w.x + l % 3 - 1;
        const int m = boxed ? deg : 0, longest = max(m, __shfl_xor(m, 32));
        for (int j = 0; j < longest; j++) {
            const int a = __shfl(at, j, 32);
            if (j < m && l < 27 && a >= 0) atomicOr(&g.cover[(a + off) >> 5], 1u << ((a + off) & 31));
        }
        lds_ready();
    }
    // This lane's cell c of round r, if it has one.
    __device__ __forceinline__ bool cell(const HashCfg& g, int r, int c, int3* q) const {
        const int l = threadIdx.x & 31;
        *q = make_int3(0, 0, 0);
        if (r >= rounds) return false;
        if (boxed) {
            const int i = 64 * r + 32 * c + l;
            if (i >= BOX_CELLS || !(lds->cover[i >> 5] >> (i & 31) & 1)) return false;
            // i is small: the quotients of i + 1/2 are far enough from whole numbers
            const int z = (int)(((float)i + 0.5f) * __builtin_amdgcn_rcpf((float)(w.x * w.y))), j = i - z * (w.x * w.y);
            const int y = (int)(((float)j + 0.5f) * __builtin_amdgcn_rcpf((float)w.x));
            *q = make_int3(lo.x + j - y * w.x, lo.y + y, lo.z + z);
            return cell_key(g, q->x, q->y, q->z) >= 0;
        }
        const int4 tc = tcell[list[r]];
        *q = around(tc, l);
        if (tc.w < 0 || l >= 27 || c) return false;
        for (int j = 0; j < r; j++)
            if (near_cell(tcell[list[j]], q->x, q->y, q->z)) return false;
        return cell_key(g, q->x, q->y, q->z) >= 0;
    }
    // Whether c is a cell around one of the triangles.
    __device__ __forceinline__ bool meets(int4 c) const {
        if (c.w < 0) return false;
        if (boxed) {
            const unsigned x = c.x - lo.x, y = c.y - lo.y, z = c.z - lo.z;
            if (x >= (unsigned)w.x || y >= (unsigned)w.y || z >= (unsigned)w.z) return false;
            const int i = ((int)z * w.y + (int)y) * w.x + (int)x;
            return rounds && (lds->cover[i >> 5] >> (i & 31) & 1);
        }
        bool in = false;
        for (int j = 0; j < deg && !in; j++) in = near_cell(tcell[list[j]], c.x, c.y, c.z);
        return in;
    }
};

// Hubs: vertices (edges) of more than HUB_FACES triangles, such as the poles of
// a sphere or the tip of a cone.  Comparing the cells around one triangle with
// those of all earlier ones, as above, is quadratic in a hub's triangles and
// done by one group (a fan of 1024 triangles, 2 units wide: 118 ms a detection).  The cells
// around a hub go into a set of its own instead, HUB_SLOTS slots per triangle
// (27 cells at most), each slot holding 27 times the place of a triangle in the
// hub's list plus a cell around it.  A unit is one triangle of one hub: 32 lanes
// enter its cells, and later visit the HUB_SLOTS slots of the set at its place,
// so that a hub's work spreads over as many groups as it has triangles (0.3 ms
// for that fan).
constexpr int HUB_SLOTS = 64;

__device__ __forceinline__ unsigned hub_slot(int3 q, unsigned slots) {
    return __umulhi(cell_slot(q.x, q.y, q.z, 0xffffffffu) * 0x9E3779B1u, slots);
}
__device__ __forceinline__ int3 hub_cell(int entry, const int* __restrict__ list, const int4* __restrict__ tcell) {
    return around(tcell[list[entry / 27]], entry % 27);
}
__device__ __forceinline__ bool same_cell(int3 a, int3 b) { return a.x == b.x && a.y == b.y && a.z == b.z; }

__global__ __launch_bounds__(256) void k_hub_count(const int* __restrict__ off, int n,
                                                   unsigned long long* __restrict__ units) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int deg = off[i + 1] - off[i];
    if (deg > HUB_FACES) atomicAdd(units, (unsigned long long)deg);
}
__global__ __launch_bounds__(256) void k_hub_units(const int* __restrict__ off, int n,
                                                   unsigned long long* __restrict__ units, int2* __restrict__ unit) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int deg = off[i + 1] - off[i];
    if (deg <= HUB_FACES) return;
    const unsigned long long at = atomicAdd(units, (unsigned long long)deg);
    for (int k = 0; k < deg; k++) unit[at + k] = make_int2(i, k);
}
// The sets of all hubs, from empty (-1) ones.
__global__ __launch_bounds__(256) void k_hub_enter(const int2* __restrict__ unit, int nunits, const int* __restrict__ off,
                                                   const int* __restrict__ tri, const int4* __restrict__ tcell,
                                                   int* __restrict__ set) {
    const int u = (int)(((long long)blockIdx.x * blockDim.x + threadIdx.x) / 32), l = threadIdx.x & 31;
    if (u >= nunits || l >= 27) return;
    const int2 h = unit[u];
    const int* list = tri + off[h.x];
    const unsigned slots = (unsigned)(off[h.x + 1] - off[h.x]) * HUB_SLOTS;
    int* own = set + (size_t)(u - h.y) * HUB_SLOTS;
    const int4 c = tcell[list[h.y]];
    if (c.w < 0) return;
    const int3 q = around(c, l);
    for (unsigned s = hub_slot(q, slots);; s = s + 1 == slots ? 0 : s + 1) {  // ends: at most 27 of 64 slots fill
        const int old = atomicCAS(&own[s], -1, h.y * 27 + l);
        if (old == -1 || same_cell(hub_cell(old, list, tcell), q)) return;
    }
}

// The cells in the slots of a unit, as CellRounds gives those of a group.
struct HubRounds {
    const int* list;
    const int4* tcell;
    const int* own;  // the hub's set
    unsigned slots, at;
    int rounds;
    __device__ __forceinline__ void start(GroupLds&, const int* list_, int deg, const int4* tcell_, const HubItem& h) {
        list = list_;
        tcell = tcell_;
        own = h.set + (size_t)(h.unit - h.place) * HUB_SLOTS;
        slots = (unsigned)deg * HUB_SLOTS;
        at = (unsigned)h.place * HUB_SLOTS;
        rounds = deg ? 1 : 0;
    }
    __device__ __forceinline__ bool cell(const HashCfg& g, int r, int c, int3* q) const {
        *q = make_int3(0, 0, 0);
        const int i = r < rounds ? own[at + 32 * c + (threadIdx.x & 31)] : -1;
        if (i < 0) return false;
        *q = hub_cell(i, list, tcell);
        return cell_key(g, q->x, q->y, q->z) >= 0;
    }
    __device__ __forceinline__ bool meets(int4 c) const {
        if (c.w < 0) return false;
        const int3 q = make_int3(c.x, c.y, c.z);
        for (unsigned s = hub_slot(q, slots);; s = s + 1 == slots ? 0 : s + 1) {
            const int i = own[s];
            if (i < 0) return false;
            if (same_cell(hub_cell(i, list, tcell), q)) return true;
        }
    }
};
static_assert(HUB_SLOTS == 64, "two slots per lane of a group");

// Vertex-face candidates by centroid cells.  Group = 32 lanes = one vertex.
// All candidates are counted; listed are all of them (LIST) or those that no
// box rules out.  Memory latency bounds it (71% of the wave cycles wait), so
// registers are held to 64 for eight waves per SIMD: 81 us against 95 with
// seven on the folded 256 x 256 cloth (5 million pairs).  Hubs are left out and
// reported; HUBS: the units of hubs instead of the nv vertices.
template <bool LIST, bool HUBS>
__global__ __launch_bounds__(64 * VISIT_WAVES, 8) void k_vf_candidates(
    HashCfg g, const float4* __restrict__ x, const float4* __restrict__ p, int nv, const int* __restrict__ vtoff,
    const int* __restrict__ vtri, const int4* __restrict__ tcell, const int* __restrict__ cnt,
    const int* __restrict__ end, unsigned mask, const FaceRec* __restrict__ ent, DetectCounts* __restrict__ c,
    int2* __restrict__ out, unsigned cap, const int2* __restrict__ unit, const int* __restrict__ hub_set) {
    __shared__ int2 buf[VISIT_WAVES][VISIT_BUF];
    __shared__ GroupLds group[VISIT_WAVES][2];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    GroupLds& lds = group[wv][lane >> 5];
    PairSink sink{buf[wv], 0, (int)((blockIdx.x * VISIT_WAVES + wv) % NEAR_BUCKETS), c, out, cap};
    int pairs = 0;
    const int stride = (int)gridDim.x * VISIT_WAVES * 2;
    for (int v0 = ((int)blockIdx.x * VISIT_WAVES + wv) * 2; v0 < nv; v0 += stride) {
        const int item = v0 + (lane >> 5), last = min(item, nv - 1);
        const int2 hub = HUBS ? unit[last] : make_int2(last, 0);
        const int v = hub.x, o = vtoff[v];
        int deg = item < nv ? vtoff[v + 1] - o : 0;
        if (!HUBS && deg > HUB_FACES) {
            c->hubs = 1;
            deg = 0;
        }
        SweptBox b = vertex_box(x[v], p[v]);
        for (int k = 0; k < 3; k++) {  // the rounding of positions between the two
            const float m = 1e-6f * fmaxf(fabsf(b.lo[k]), fabsf(b.hi[k]));
            b.lo[k] -= m;
            b.hi[k] += m;
        }
        std::conditional_t<HUBS, HubRounds, CellRounds> cells;
        cells.start(lds, vtri + o, deg, tcell, HubItem{hub_set, last, hub.y});
        const int rounds = max(cells.rounds, __shfl_xor(cells.rounds, 32));
        for (int r = 0; r < rounds; r++) {
            int3 q[2];
            int start[2], n[2];
            if (!__any(cell_runs(cells, g, r, cnt, end, mask, q, start, n))) continue;
            visit_runs(lds, q, start, n, [&](int e, int3 fq) {
                bool hit = false;
                int f = 0;
                if (e >= 0) {
                    const FaceRec rec = ent[e];
                    f = rec.face;
                    // a slot may hold other cells' faces too
                    if (rec.cx == fq.x && rec.cy == fq.y && rec.cz == fq.z && v != rec.v0 && v != rec.v1 && v != rec.v2) {
                        pairs++;
                        hit = LIST || !(rec.cull && box_misses(b, rec));
                    }
                }
                sink.add(hit, v, f);
            });
        }
    }
    if (sink.n) sink.flush();
    if (!LIST) sink.count(pairs);
}

// Vertex-face candidates by swept boxes: the faces entered in the cells of the
// vertex's box, level by level, taken at the lowest cell that the two boxes'
// cell ranges share.
__global__ __launch_bounds__(64 * VISIT_WAVES) void k_swept_candidates(
    HashCfg g, HashCfg gi, const float4* __restrict__ x, const float4* __restrict__ p, int nv,
    const int* __restrict__ vtoff, const int* __restrict__ cnt, const int* __restrict__ end, unsigned mask,
    const int2* __restrict__ ent, unsigned ent_cap, const FaceRec* __restrict__ rec, const int4* __restrict__ fcell,
    DetectCounts* __restrict__ c, int2* __restrict__ out, unsigned cap) {
    __shared__ int2 buf[VISIT_WAVES][VISIT_BUF];
    __shared__ GroupLds group[VISIT_WAVES][2];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, l = lane & 31;
    PairSink sink{buf[wv], 0, (int)((blockIdx.x * VISIT_WAVES + wv) % NEAR_BUCKETS), c, out, cap};
    int pairs = 0;
    unsigned levels = 0;  // that hold faces, the same for all
    for (int k = 0; k < SWEPT_LEVELS; k++) levels |= c->level[k] ? 1u << k : 0u;
    const int stride = (int)gridDim.x * VISIT_WAVES * 2;
    for (int v0 = ((int)blockIdx.x * VISIT_WAVES + wv) * 2; v0 < nv; v0 += stride) {
        const int v = v0 + (lane >> 5), at = min(v, nv - 1);
        const bool used = v < nv && vtoff[at + 1] > vtoff[at];
        const SweptBox b = vertex_box(x[at], p[at]);
        long long span = 1;
        for (int k = 0; k < 3; k++)
            span *= (long long)min(cell_coord(g, b.hi[k], k) - cell_coord(g, b.lo[k], k) + 1, SWEPT_MAX_CELLS + 1);
        const bool over = span > SWEPT_MAX_CELLS;
        if (used && over) c->vertex_span = 1;
        float scale = 1.0f;
        for (int level = 0; level < SWEPT_LEVELS; level++, scale *= (float)SWEPT_FACTOR) {
            if (!(levels >> level & 1)) continue;
            int lo[3], w[3];
            for (int k = 0; k < 3; k++) {
                lo[k] = cell_coord(gi, b.lo[k], k, scale);
                w[k] = min(cell_coord(gi, b.hi[k], k, scale) - lo[k] + 1, SWEPT_MAX_CELLS + 1);
            }
            const int cells = used && !over ? w[0] * w[1] * w[2] : 0;
            // cells of the box may agree in their codes
            const bool wide = w[0] >= CODE_SPAN || w[1] >= CODE_SPAN || w[2] >= CODE_SPAN;
            auto cell_of = [&](int i) { return make_int3(lo[0] + i % w[0], lo[1] + i / w[0] % w[1], lo[2] + i / (w[0] * w[1])); };
            const int most = max(cells, __shfl_xor(cells, 32));
            for (int c0 = 0; c0 < most; c0 += 64) {
                int3 q[2];
                int start[2], n[2];
                for (int c = 0; c < 2; c++) {
                    const bool mine = c0 + 32 * c + l < cells;
                    q[c] = cell_of(c0 + 32 * c + l);
                    const unsigned slot = mine ? level_slot(q[c].x, q[c].y, q[c].z, level, mask) : 0u;
                    const int m = cnt[slot], e1 = end[slot];
                    n[c] = mine && (unsigned)e1 <= ent_cap ? m : 0;  // beyond: the table did not fit, the caller starts over
                    start[c] = e1 - m;
                }
                visit_runs(group[wv][lane >> 5], q, start, n, [&](int e, int3 fq) {
                    bool hit = false;
                    int f = 0;
                    if (e >= 0) {
                        const int2 en = ent[e];
                        f = en.x;
                        bool in = (en.y & 0x7ffffff) == cell_code(fq.x, fq.y, fq.z) &&
                                  (int)((unsigned)en.y >> 30) == level && ((en.y >> 27 & 1) || fq.x == lo[0]) &&
                                  ((en.y >> 28 & 1) || fq.y == lo[1]) && ((en.y >> 29 & 1) || fq.z == lo[2]);
                        if (wide && in) {
                            const int4 a = fcell[2 * f], z = fcell[2 * f + 1];
                            in = fq.x >= a.x && fq.x <= z.x && fq.y >= a.y && fq.y <= z.y && fq.z >= a.z && fq.z <= z.z;
                        }
                        if (in) {
                            const FaceRec r = rec[f];
                            hit = !box_misses(b, r) && v != r.v0 && v != r.v1 && v != r.v2;
                            pairs += hit;
                        }
                    }
                    sink.add(hit, v, f);
                });
            }
        }
    }
    if (sink.n) sink.flush();
    sink.count(pairs);
}

// Whether two edges' swept boxes lie further apart along an axis than the
// contact distance and the rounding of the closest points' coordinates: every
// point the narrowphase measures between lies in the boxes, so such a pair is
// no contact.  (False for NaN.)
__device__ __forceinline__ bool edges_apart(const SweptBox& a, const SweptBox& b, float th) {
    auto apart = [&](float hi, float lo) { return lo - hi > 2.0f * th + 2e-6f * (fabsf(lo) + fabsf(hi)); };
    bool r = false;
    for (int k = 0; k < 3; k++) r = r || apart(a.hi[k], b.lo[k]) || apart(b.hi[k], a.lo[k]);
    return r;
}

// An entry of the edge table: an edge in one of the cells of its faces, with
// its ends and the swept box of the four points, not widened.  `before`: none
// (0), one (1: the cell o) or several (2) of the edge's other cells come first
// in the order of its faces.  EDGE_HUB: an edge of more than HUB_FACES faces,
// entered once per face, ox its place in etri; telling its distinct cells apart
// one by one took 0.3 s for 1024 faces.
constexpr int EDGE_HUB = 4;
struct alignas(64) EdgeRec {
    int cx, cy, cz, edge;
    int v0, v1, before, ox;
    int oy, oz;
    SweptBox box;
};

// Calls f(e, cell, before, other) for every entry of this lane's edge e (0 <= e
// < ne), a hub's by all lanes of the wave.  Called by all of them.
template <class F>
__device__ __forceinline__ void edge_cells(int e, int ne, const int* __restrict__ etoff, const int* __restrict__ etri,
                                           const int4* __restrict__ tcell, F&& f) {
    int o = 0, deg = 0;
    if (e < ne) {
        o = etoff[e];
        deg = etoff[e + 1] - o;
    }
    for (unsigned long long hubs = __ballot(deg > HUB_FACES); hubs; hubs &= hubs - 1) {
        const int lane = __ffsll(hubs) - 1, h = __shfl(e, lane), h0 = __shfl(o, lane), h1 = h0 + __shfl(deg, lane);
        for (int j = h0 + (int)(threadIdx.x & 63); j < h1; j += 64) {
            const int4 c = tcell[etri[j]];
            if (c.w >= 0) f(h, c, EDGE_HUB, make_int4(j, 0, 0, 0));
        }
    }
    if (deg > HUB_FACES) return;
    int4 other = make_int4(0, 0, 0, 0);
    int distinct = 0;
    for (int j = 0; j < deg; j++) {
        const int4 c = tcell[etri[o + j]];
        bool fresh = c.w >= 0;
        for (int m = 0; m < j && fresh; m++) {
            const int4 d = tcell[etri[o + m]];
            fresh = d.w < 0 || d.x != c.x || d.y != c.y || d.z != c.z;
        }
        if (!fresh) continue;
        f(e, c, min(distinct, 2), other);
        if (!distinct++) other = c;
    }
}

__global__ __launch_bounds__(256) void k_tri_cells(HashCfg g, const float4* __restrict__ p, const int* __restrict__ tris,
                                                   int nt, unsigned mask, int4* __restrict__ tcell) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nt) return;
    int gp[3];
    tri_cell(g, p, tris, t, gp);
    const bool in = cell_key(g, gp[0], gp[1], gp[2]) >= 0;
    tcell[t] = make_int4(gp[0], gp[1], gp[2], in ? (int)cell_slot(gp[0], gp[1], gp[2], mask) : -1);
}

__global__ __launch_bounds__(256) void k_edge_count(int ne, const int* __restrict__ etoff, const int* __restrict__ etri,
                                                    const int4* __restrict__ tcell, int* __restrict__ cnt) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    edge_cells(e, ne, etoff, etri, tcell, [&](int, int4 c, int, int4) { atomicAdd(&cnt[c.w], 1); });
}

// Each entry takes the next place of its slot, so that place[] ends at the
// slots' ends.
__global__ __launch_bounds__(256) void k_edge_fill(int ne, const int2* __restrict__ edges, const int* __restrict__ etoff,
                                                   const int* __restrict__ etri, const int4* __restrict__ tcell,
                                                   const float4* __restrict__ x, const float4* __restrict__ p,
                                                   int* __restrict__ place, EdgeRec* __restrict__ ent) {
    const int mine = blockIdx.x * blockDim.x + threadIdx.x;
    edge_cells(mine, ne, etoff, etri, tcell, [&](int e, int4 c, int before, int4 o) {
        const int2 v = edges[e];
        SweptBox b = vertex_box(x[v.x], p[v.x]);
        box_add(b, x[v.y]);
        box_add(b, p[v.y]);
        ent[atomicAdd(&place[c.w], 1)] = EdgeRec{c.x, c.y, c.z, e, v.x, v.y, before, o.x, o.y, o.z, b};
    });
}

// Edge-edge candidates (new: the reference declares Contact::EE, CCD_Basic.h:14,
// and leaves it unimplemented, CCD.cpp:925-928): every pair of edges of two
// triangles whose centroid cells are at most one cell apart that shares no
// vertex and has no vertex that is a mesh neighbour of the other edge's (pairs
// that close in the mesh are material neighbours, not contacts), once, as
// (lower edge id, higher edge id).  Group = 32 lanes = the lower edge a: the
// cells around its triangles, each once; an edge b entered in several of them
// counts at the first in the order of its faces.
// Edges have entries of their own, with all that the tests read: visiting the
// faces' entries instead offered most edges twice and took four dependent
// gathers to tell (fold of 96 x 96: 151 us against 84).  Hubs are left out and
// reported; HUBS: the units of hubs instead of the ne edges.
constexpr int RING_MAX = 64;

// Whether id is among n neighbours, which are in ascending order beyond RING_SORTED.
constexpr int RING_SORTED = 16;
__device__ __forceinline__ bool listed(const int* __restrict__ a, int n, int id) {
    if (n > RING_SORTED) {
        int lo = 0;  // the last one not above id, if any
        for (int len = n; len > 1; len -= len / 2)
            if (a[lo + len / 2] <= id) lo += len / 2;
        return a[lo] == id;
    }
    bool in = false;
    for (int i = 0; i < n; i++) in |= a[i] == id;
    return in;
}

template <bool LIST, bool HUBS>
__global__ __launch_bounds__(64 * VISIT_WAVES) void k_ee_candidates(
    HashCfg g, int ne, const int2* __restrict__ edges, const int* __restrict__ etoff, const int* __restrict__ etri,
    const int* __restrict__ voff, const int* __restrict__ vnbr, const float4* __restrict__ x,
    const float4* __restrict__ p, const int4* __restrict__ tcell, const int* __restrict__ cnt,
    const int* __restrict__ end, unsigned mask, const EdgeRec* __restrict__ ent, float th, DetectCounts* __restrict__ c,
    int2* __restrict__ out, unsigned cap, const int2* __restrict__ unit, const int* __restrict__ hub_set) {
    __shared__ int2 buf[VISIT_WAVES][VISIT_BUF];
    __shared__ int4 ring_s[VISIT_WAVES][2][RING_MAX / 4];
    __shared__ GroupLds group[VISIT_WAVES][2];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, l = lane & 31;
    GroupLds& lds = group[wv][lane >> 5];
    int4* ring = ring_s[wv][lane >> 5];
    PairSink sink{buf[wv], 0, (int)((blockIdx.x * VISIT_WAVES + wv) % NEAR_BUCKETS), c, out, cap};
    int pairs = 0;
    const int stride = (int)gridDim.x * VISIT_WAVES * 2;
    for (int a0 = ((int)blockIdx.x * VISIT_WAVES + wv) * 2; a0 < ne; a0 += stride) {
        const int item = a0 + (lane >> 5), last = min(item, ne - 1);
        const int2 hub = HUBS ? unit[last] : make_int2(last, 0);
        const int a = hub.x, o = etoff[a];
        const int2 av = edges[a];
        int deg = item < ne ? etoff[a + 1] - o : 0;
        if (!HUBS && deg > HUB_FACES) {
            c->hubs = 1;
            deg = 0;
        }
        SweptBox abox = vertex_box(x[av.x], p[av.x]);
        box_add(abox, x[av.y]);
        box_add(abox, p[av.y]);
        // a's vertices and their mesh neighbours: an edge with a vertex among them is no candidate
        const int r0 = voff[av.x], n0 = voff[av.x + 1] - r0, r1 = voff[av.y], n1 = voff[av.y + 1] - r1;
        const int quads = (n0 + n1 + 5) / 4;
        const bool fits = quads <= RING_MAX / 4;
        __builtin_amdgcn_wave_barrier();  // the edge before is done with the lists
        if (fits)
            for (int i = l; i < 4 * quads; i += 32)
                reinterpret_cast<int*>(ring)[i] = i == 0            ? av.x
                                                  : i == 1          ? av.y
                                                  : i < n0 + 2      ? vnbr[r0 + i - 2]
                                                  : i < n0 + n1 + 2 ? vnbr[r1 + i - 2 - n0]
                                                                    : -1;
        std::conditional_t<HUBS, HubRounds, CellRounds> cells;
        cells.start(lds, etri + o, deg, tcell, HubItem{hub_set, last, hub.y});
        auto ringed = [&](int u, int w) {
            bool in = false;
            if (fits) {
                for (int i = 0; i < quads; i++) {
                    const int4 r = ring[i];
                    in |= r.x == u || r.y == u || r.z == u || r.w == u || r.x == w || r.y == w || r.z == w || r.w == w;
                }
                return in;
            }
            return u == av.x || u == av.y || w == av.x || w == av.y || listed(vnbr + r0, n0, u) ||
                   listed(vnbr + r0, n0, w) || listed(vnbr + r1, n1, u) || listed(vnbr + r1, n1, w);
        };
        const int rounds = max(cells.rounds, __shfl_xor(cells.rounds, 32));
        for (int r = 0; r < rounds; r++) {
            int3 q[2];
            int start[2], n[2];
            if (!__any(cell_runs(cells, g, r, cnt, end, mask, q, start, n))) continue;
            visit_runs(lds, q, start, n, [&](int e, int3 fq) {
                bool hit = false;
                int eb = 0;
                if (e >= 0) {
                    const EdgeRec rec = ent[e];
                    eb = rec.edge;
                    if (eb > a && rec.cx == fq.x && rec.cy == fq.y && rec.cz == fq.z && !ringed(rec.v0, rec.v1)) {
                        bool first = !(rec.before & 3) || !cells.meets(make_int4(rec.ox, rec.oy, rec.oz, 0));
                        if (rec.before >= 2) {
                            const int own = rec.before == EDGE_HUB ? rec.ox : INT_MAX;
                            for (int j = etoff[eb]; first && j != own; j++) {  // ends at a face of this cell
                                const int4 d = tcell[etri[j]];
                                if (own == INT_MAX && d.w >= 0 && d.x == rec.cx && d.y == rec.cy && d.z == rec.cz) break;
                                first = !cells.meets(d);
                            }
                        }
                        pairs += first;
                        hit = first && (LIST || !edges_apart(abox, rec.box, th));
                    }
                }
                sink.add(hit, a, eb);
            });
        }
    }
    if (sink.n) sink.flush();
    if (!LIST) sink.count(pairs);
}

// Vertex -> triangles (CSR, any order within a vertex).
__global__ __launch_bounds__(256) void k_vt_count(const int* __restrict__ tris, int n, int* __restrict__ cnt) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) atomicAdd(&cnt[tris[i]], 1);
}
__global__ __launch_bounds__(256) void k_vt_fill(const int* __restrict__ tris, int n, const int* __restrict__ off,
                                                 int* __restrict__ cnt, int* __restrict__ vtri) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) vtri[off[tris[i]] + atomicSub(&cnt[tris[i]], 1) - 1] = i / 3;
}
// The bucketed list as two arrays; at[b]: where bucket b's pairs go.
struct BucketPlaces {
    int at[NEAR_BUCKETS + 1];
};
__global__ __launch_bounds__(256) void k_unzip(const int2* __restrict__ a, unsigned cap, BucketPlaces b,
                                               uint32_t* __restrict__ hi, uint32_t* __restrict__ lo) {
    const int n = b.at[blockIdx.y + 1] - b.at[blockIdx.y];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int2 q = a[(size_t)blockIdx.y * cap + i];
    hi[b.at[blockIdx.y] + i] = (uint32_t)q.x;
    lo[b.at[blockIdx.y] + i] = (uint32_t)q.y;
}

// ---------------------------------------------------------------------------
// narrowphase: FP64 cubic (solve_cubic / newtons_method / solve_quadratic,
// CCD.cpp:48-113), ExtendedVFTest (CCD.cpp:1733-1808)
// ---------------------------------------------------------------------------
__device__ int d_solve_quadratic(double a, double b, double c, double* x) {
    double d = b * b - 4 * a * c;
    if (d < 0) {
        x[0] = -b / (2 * a);
        return 0;
    }
    double q = -(b + (b < 0 ? -1.0 : 1.0) * sqrt(d)) / 2;
    int i = 0;
    if (fabs(a) > 1e-12 * fabs(q)) x[i++] = q / a;
    if (fabs(q) > 1e-12 * fabs(c)) x[i++] = c / q;
    if (i == 2 && x[0] > x[1]) {
        double t = x[0];
        x[0] = x[1];
        x[1] = t;
    }
    return i;
}

__device__ double d_newton(double a, double b, double c, double d, double x0, int init_dir) {
    if (init_dir != 0) {
        double y0 = d + x0 * (c + x0 * (b + x0 * a));
        double ddy0 = 2 * b + x0 * (6 * a);
        x0 += init_dir * sqrt(fabs(2 * y0 / ddy0));
    }
    for (int iter = 0; iter < 100; iter++) {
        double y = d + x0 * (c + x0 * (b + x0 * a));
        double dy = c + x0 * (2 * b + x0 * 3 * a);
        if (dy == 0) return x0;
        double x1 = x0 - y / dy;
        if (fabs(x0 - x1) < 1e-6) return x0;
        x0 = x1;
    }
    return x0;
}

// When the critical-point quadratic leaves its root unset (a = b = 0: the
// cubic is linear; the reference reads an unset value there), Newton starts
// from 0, which converges to the linear root.
__device__ int d_solve_cubic(double a, double b, double c, double d, double* x) {
    double xc[2];
    xc[0] = __longlong_as_double(0x7ff8000000000000ll);
    xc[1] = xc[0];
    int ncrit = d_solve_quadratic(3 * a, 2 * b, c, xc);
    if (ncrit == 0) {
        if (xc[0] != xc[0]) xc[0] = 0.0;
        x[0] = d_newton(a, b, c, d, xc[0], 0);
        return 1;
    } else if (ncrit == 1) {
        return d_solve_quadratic(b, c, d, x);
    }
    double yc0 = d + xc[0] * (c + xc[0] * (b + xc[0] * a)), yc1 = d + xc[1] * (c + xc[1] * (b + xc[1] * a));
    int i = 0;
    if (yc0 * a >= 0) x[i++] = d_newton(a, b, c, d, xc[0], -1);
    if (yc0 * yc1 <= 0) {
        int closer = fabs(yc0) < fabs(yc1) ? 0 : 1;
        x[i++] = d_newton(a, b, c, d, xc[closer], closer == 0 ? 1 : -1);
    }
    if (yc1 * a <= 0) x[i++] = d_newton(a, b, c, d, xc[1], 1);
    return i;
}

__device__ __forceinline__ V3 v3(float4 a) { return mk(a.x, a.y, a.z); }
__device__ __forceinline__ V3 vnormalize(V3 a) {
    float inv = 1.0f / sqrtf(dot(a, a));
    return V3{a.x * inv, a.y * inv, a.z * inv};
}
__device__ __forceinline__ float stp(V3 u, V3 v, V3 w) { return dot(u, cross(v, w)); }
__device__ __forceinline__ V3 lerp(V3 x, V3 p, double t) {
    float tf = (float)t;
    return V3{x.x + tf * (p.x - x.x), x.y + tf * (p.y - x.y), x.z + tf * (p.z - x.z)};
}
// BarycentricCoord (CCD.cpp:115-130)
__device__ __forceinline__ V3 bary(V3 pp, V3 a, V3 b, V3 c) {
    V3 AB = sub(a, c), AC = sub(b, c), AP = sub(pp, c);
    float d00 = dot(AC, AC), d01 = dot(AC, AB), d02 = dot(AC, AP), d11 = dot(AB, AB), d12 = dot(AB, AP);
    float inv = 1 / (d00 * d11 - d01 * d01);
    float v = (d11 * d02 - d01 * d12) * inv;
    float u = (d00 * d12 - d01 * d02) * inv;
    float w = 1 - u - v;
    return V3{u, v, w};
}
__device__ __forceinline__ float dist3(V3 a, V3 b) {
    V3 d = sub(a, b);
    return sqrtf(d.x * d.x + d.y * d.y + d.z * d.z);
}

__device__ bool vf_ccd(V3 x0, V3 x1, V3 x2, V3 x3, V3 p0, V3 p1, V3 p2, V3 p3, float th, float* t_out, V3* n_out,
                       V3* w_out) {
    V3 v0 = sub(p0, x0);
    V3 X1 = sub(x1, x0), X2 = sub(x2, x0), X3 = sub(x3, x0);
    V3 V1 = sub(sub(p1, x1), v0), V2 = sub(sub(p2, x2), v0), V3_ = sub(sub(p3, x3), v0);
    double a0 = stp(X1, X2, X3);
    double a1 = (double)(stp(V1, X2, X3) + stp(X1, V2, X3) + stp(X1, X2, V3_));
    double a2 = (double)(stp(X1, V2, V3_) + stp(V1, X2, V3_) + stp(V1, V2, X3));
    double a3 = stp(V1, V2, V3_);
    double t[5];
    int nsol = d_solve_cubic(a3, a2, a1, a0, t);
    int m = 0;
    for (int i = 0; i < nsol; i++)
        if (isfinite(t[i])) t[m++] = t[i];
    t[m] = 1;
    t[m + 1] = 0;
    int nt = m + 2;
    for (int i = 1; i < nt; i++) {
        double v = t[i];
        int j = i - 1;
        while (j >= 0 && t[j] > v) {
            t[j + 1] = t[j];
            j--;
        }
        t[j + 1] = v;
    }
    for (int i = 0; i < nt; i++) {
        if (t[i] < 0 || t[i] > 1) continue;
        V3 c0 = lerp(x0, p0, t[i]), c1 = lerp(x1, p1, t[i]), c2 = lerp(x2, p2, t[i]), c3 = lerp(x3, p3, t[i]);
        V3 nrm = vnormalize(cross(sub(p2, p1), sub(p3, p1)));
        V3 cn = vnormalize(cross(sub(c2, c1), sub(c3, c1)));
        double dist = dot(sub(c0, c1), cn);
        V3 wg = bary(c0, c1, c2, c3);
        float ed1 = dist3(c1, c2), ed2 = dist3(c1, c3), ed3 = dist3(c2, c3);
        float eps = th / ((ed1 + ed2 + ed3) / 3.0);
        bool in1 = (wg.x <= (1 + eps)) && (wg.x >= (-eps));
        bool in2 = (wg.y <= (1 + eps)) && (wg.y >= (-eps));
        bool in3 = (wg.z <= (1 + eps)) && (wg.z >= (-eps));
        if ((fabs(dist) - 2.0f * th < -1e-6) && in1 && in2 && in3) {
            *t_out = (float)t[i];
            *n_out = nrm;
            *w_out = wg;
            return true;
        }
    }
    return false;
}

// This workgroup's share of the bucketed candidate list: bucket blockIdx.x %
// NEAR_BUCKETS, pairs from `from` on in steps of `step`.
struct NearRun {
    const int2* pairs;
    unsigned n, from, step;
    __device__ __forceinline__ NearRun(const int2* near, unsigned cap, const DetectCounts* c) {
        const unsigned b = blockIdx.x % NEAR_BUCKETS;
        pairs = near + (size_t)b * cap;
        n = min(c->bucket[b].near, cap);
        from = blockIdx.x / NEAR_BUCKETS * 256;
        step = gridDim.x / NEAR_BUCKETS * 256;
    }
};

// The narrowphase over the listed pairs (their number is on the device), its
// contacts appended in any order.  STORE: time, normal and weights too (the
// response needs only the vertices).  Pairs outside the face's half-spaces are
// dropped first, and the workgroup gathers the others until it has one for
// every thread, since the cubic is some 3000 instructions (folded 256 x 256
// cloth: 17,000 of 1.1 million pairs are left; 160 us without the half-spaces,
// 33 with them; 14.3 million swept-box pairs of a 512 x 512 one: 970 and 138).
template <bool STORE>
__global__ __launch_bounds__(256) void k_narrow(const int2* __restrict__ near, unsigned near_cap,
                                                const int* __restrict__ tris, const FaceAxes* __restrict__ axes,
                                                const float4* __restrict__ x, const float4* __restrict__ p, float th,
                                                DetectCounts* __restrict__ c, unsigned cap, int4* __restrict__ vquad,
                                                int2* __restrict__ vf, float* __restrict__ ct, float* __restrict__ cn,
                                                double* __restrict__ cw) {
    __shared__ int2 left[512];
    __shared__ unsigned left_n;
    if (threadIdx.x == 0) left_n = 0;
    __syncthreads();
    const NearRun run(near, near_cap, c);
    auto solve = [&](int2 q) {
        const int4 v = make_int4(q.x, tris[3 * q.y], tris[3 * q.y + 1], tris[3 * q.y + 2]);
        float t;
        V3 nr, wg;
        if (!vf_ccd(v3(x[v.x]), v3(x[v.y]), v3(x[v.z]), v3(x[v.w]), v3(p[v.x]), v3(p[v.y]), v3(p[v.z]), v3(p[v.w]), th,
                    &t, &nr, &wg))
            return;
        const unsigned o = atomicAdd(&c->contacts, 1u);
        if (o >= cap) return;
        vquad[o] = v;
        if (STORE) {
            vf[o] = q;
            ct[o] = t;
            cn[3 * o] = nr.x;
            cn[3 * o + 1] = nr.y;
            cn[3 * o + 2] = nr.z;
            cw[4 * o] = 1.0;
            cw[4 * o + 1] = wg.x;
            cw[4 * o + 2] = wg.y;
            cw[4 * o + 3] = wg.z;
        }
    };
    for (unsigned i0 = run.from; i0 < run.n; i0 += run.step) {
        const unsigned i = i0 + threadIdx.x;
        const bool last = i0 + run.step >= run.n;
        int2 q = make_int2(0, 0);
        bool keep = i < run.n;
        if (keep) {
            q = run.pairs[i];
            keep = !axes_miss(axes[q.y], x[q.x], p[q.x]);
        }
        if (keep) left[atomicAdd(&left_n, 1u)] = q;
        __syncthreads();
        const unsigned n = left_n;
        __syncthreads();  // every thread has read it before it changes
        if (n < 256 && !last) continue;
        for (unsigned k = threadIdx.x; k < n; k += 256) solve(left[k]);
        __syncthreads();
        if (threadIdx.x == 0) left_n = 0;
        __syncthreads();
    }
}

// Contacts in ascending (first, second) order, for callers that read them:
// counted by their first id, scanned, dealt to their first id's run, and each
// placed by the number of smaller second ids in its run.
__global__ __launch_bounds__(256) void k_first_count(const int2* __restrict__ key, int n, int* __restrict__ cnt) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) atomicAdd(&cnt[key[i].x], 1);
}
__global__ __launch_bounds__(256) void k_first_deal(const int2* __restrict__ key, int n, const int* __restrict__ off,
                                                    int* __restrict__ cnt, int* __restrict__ idx) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) idx[off[key[i].x] + atomicSub(&cnt[key[i].x], 1) - 1] = i;
}
__global__ __launch_bounds__(256) void k_contact_order(const int2* __restrict__ key, int n, const int* __restrict__ off,
                                                       const int* __restrict__ idx, const float* __restrict__ t,
                                                       const float* __restrict__ nr, const double* __restrict__ w,
                                                       const int4* __restrict__ quad, int2* __restrict__ okey,
                                                       float* __restrict__ ot, float* __restrict__ on,
                                                       double* __restrict__ ow, int4* __restrict__ oquad) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int2 k = key[i];
    int at = off[k.x];
    for (int j = off[k.x]; j < off[k.x + 1]; j++) at += key[idx[j]].y < k.y;
    okey[at] = k;
    ot[at] = t[i];
    for (int a = 0; a < 3; a++) on[3 * at + a] = nr[3 * i + a];
    for (int a = 0; a < 4; a++) ow[4 * at + a] = w[4 * i + a];
    if (quad) oquad[at] = quad[i];
}

// ---------------------------------------------------------------------------
// edge-edge narrowphase and response (new; see k_ee_candidates)
// ---------------------------------------------------------------------------
__device__ __forceinline__ long long to_fixed(float f) { return (long long)rint((double)f * 4294967296.0); }
__device__ __forceinline__ float clamp01(float v) { return v < 0.0f ? 0.0f : (v > 1.0f ? 1.0f : v); }

// Closest points a0 + s (a1 - a0), b0 + u (b1 - b0), s, u in [0, 1], of two
// segments (Ericson 2005, Real-Time Collision Detection, sec. 5.1.9).
__device__ void seg_closest(V3 a0, V3 a1, V3 b0, V3 b1, float* s_out, float* u_out) {
    V3 d1 = sub(a1, a0), d2 = sub(b1, b0), r = sub(a0, b0);
    float a = dot(d1, d1), e = dot(d2, d2), f = dot(d2, r);
    float s, u;
    if (a <= 1e-30f && e <= 1e-30f) {
        s = 0.0f;
        u = 0.0f;
    } else if (a <= 1e-30f) {
        s = 0.0f;
        u = clamp01(f / e);
    } else {
        float c = dot(d1, r);
        if (e <= 1e-30f) {
            u = 0.0f;
            s = clamp01(-c / a);
        } else {
            float b = dot(d1, d2);
            float den = a * e - b * b;
            s = den > 0.0f ? clamp01((b * f - c * e) / den) : 0.0f;
            u = (b * s + f) / e;
            if (u < 0.0f) {
                u = 0.0f;
                s = clamp01(-c / a);
            } else if (u > 1.0f) {
                u = 1.0f;
                s = clamp01((b - c) / a);
            }
        }
    }
    *s_out = s;
    *u_out = u;
}

__device__ __forceinline__ V3 seg_point(V3 a0, V3 a1, float s) {
    return V3{a0.x + s * (a1.x - a0.x), a0.y + s * (a1.y - a0.y), a0.z + s * (a1.z - a0.z)};
}

// Whether two edges can be in contact: not near parallel (sin^2 of the
// angle > 1e-12) and, at the start of the step, at least one thickness apart
// along the normal n of the edges (q1 - q0) x (q3 - q2).  Edges that start
// side by side (neighbours in one sheet whose spacing is below the contact
// gap) have no separation along n to restore and are not contacts.
__device__ bool ee_separable(V3 X0, V3 X1, V3 X2, V3 X3, V3 q0, V3 q1, V3 q2, V3 q3, float th, V3* side_out,
                             V3* n_out) {
    float s0, u0;
    seg_closest(X0, X1, X2, X3, &s0, &u0);
    V3 side = sub(seg_point(X0, X1, s0), seg_point(X2, X3, u0));
    V3 ea = sub(q1, q0), eb = sub(q3, q2);
    V3 cr = cross(ea, eb);
    if (dot(cr, cr) <= 1e-12f * (dot(ea, ea) * dot(eb, eb))) return false;
    V3 nn = vnormalize(cr);
    if (!(fabsf(dot(side, nn)) >= th)) return false;
    *side_out = side;
    *n_out = nn;
    return true;
}

// Edge (x0, x1) -> (p0, p1) against edge (x2, x3) -> (p2, p3) over the step,
// for separable edges (ee_separable at the end state): the times the four
// points are coplanar (the cubic of vf_ccd, with the first edge's start
// point as origin; Provot 1997) plus t = 0 and 1, ascending; the first time
// in [0, 1] where the segments come within 2 x thickness is the contact.
// Records t, the end-state edge normal (p1 - p0) x (p3 - p2) normalised and
// the weights (1 - s, s, 1 - u, u) of the closest points.
__device__ bool ee_ccd(V3 x0, V3 x1, V3 x2, V3 x3, V3 p0, V3 p1, V3 p2, V3 p3, float th, float* t_out, V3* n_out,
                       float* w_out) {
    V3 side, nrm;
    if (!ee_separable(x0, x1, x2, x3, p0, p1, p2, p3, th, &side, &nrm)) return false;
    V3 v0 = sub(p0, x0);
    V3 X1 = sub(x1, x0), X2 = sub(x2, x0), X3 = sub(x3, x0);
    V3 V1 = sub(sub(p1, x1), v0), V2 = sub(sub(p2, x2), v0), V3_ = sub(sub(p3, x3), v0);
    double a0 = stp(X1, X2, X3);
    double a1 = (double)(stp(V1, X2, X3) + stp(X1, V2, X3) + stp(X1, X2, V3_));
    double a2 = (double)(stp(X1, V2, V3_) + stp(V1, X2, V3_) + stp(V1, V2, X3));
    double a3 = stp(V1, V2, V3_);
    double t[5];
    int nsol = d_solve_cubic(a3, a2, a1, a0, t);
    int m = 0;
    for (int i = 0; i < nsol; i++)
        if (isfinite(t[i])) t[m++] = t[i];
    t[m] = 1;
    t[m + 1] = 0;
    int nt = m + 2;
    for (int i = 1; i < nt; i++) {
        double v = t[i];
        int j = i - 1;
        while (j >= 0 && t[j] > v) {
            t[j + 1] = t[j];
            j--;
        }
        t[j + 1] = v;
    }
    for (int i = 0; i < nt; i++) {
        if (t[i] < 0 || t[i] > 1) continue;
        V3 c0 = lerp(x0, p0, t[i]), c1 = lerp(x1, p1, t[i]), c2 = lerp(x2, p2, t[i]), c3 = lerp(x3, p3, t[i]);
        float s, u;
        seg_closest(c0, c1, c2, c3, &s, &u);
        float d = dist3(seg_point(c0, c1, s), seg_point(c2, c3, u));
        if (d - 2.0f * th < -1e-6f) {
            *t_out = (float)t[i];
            *n_out = nrm;
            w_out[0] = 1.0f - s;
            w_out[1] = s;
            w_out[2] = 1.0f - u;
            w_out[3] = u;
            return true;
        }
    }
    return false;
}

template <bool STORE>
__global__ __launch_bounds__(256) void k_narrow_ee(const int2* __restrict__ near, unsigned near_cap,
                                                   const int2* __restrict__ edges, const float4* __restrict__ x,
                                                   const float4* __restrict__ p, float th, DetectCounts* __restrict__ c,
                                                   unsigned cap, int2* __restrict__ ab, int4* __restrict__ quad,
                                                   float* __restrict__ ct, float* __restrict__ cn,
                                                   double* __restrict__ cw) {
    const NearRun run(near, near_cap, c);
    for (unsigned i = run.from + threadIdx.x; i < run.n; i += run.step) {
        const int2 q = run.pairs[i];
        const int2 ea = edges[q.x], eb = edges[q.y];
        float t, w[4];
        V3 nr;
        if (!ee_ccd(v3(x[ea.x]), v3(x[ea.y]), v3(x[eb.x]), v3(x[eb.y]), v3(p[ea.x]), v3(p[ea.y]), v3(p[eb.x]),
                    v3(p[eb.y]), th, &t, &nr, w))
            continue;
        const unsigned o = atomicAdd(&c->contacts, 1u);
        if (o >= cap) continue;
        quad[o] = make_int4(ea.x, ea.y, eb.x, eb.y);
        if (STORE) {
            ab[o] = q;
            ct[o] = t;
            cn[3 * o] = nr.x;
            cn[3 * o + 1] = nr.y;
            cn[3 * o + 2] = nr.z;
            for (int k = 0; k < 4; k++) cw[4 * o + k] = w[k];
        }
    }
}

// Edge-edge response on the current positions, for separable edges
// (ee_separable): the closest points of the two edges are pushed apart along
// the edge normal (oriented as the closest points' offset at the start of
// the step) until they are 2 x thickness apart, half each, spread over each
// edge's ends by the closest-point weights (w_k / sum w^2, so the closest
// point moves by the full half); a static edge leaves the whole gap to the
// other.  Fixes are summed in the vertex-face response's fixed-point
// accumulators.
__device__ bool ee_fix(const V3* X, const V3* q, float th, V3* d) {
    V3 side, nn;
    if (!ee_separable(X[0], X[1], X[2], X[3], q[0], q[1], q[2], q[3], th, &side, &nn)) return false;
    if (dot(side, nn) < 0.0f) nn = V3{-nn.x, -nn.y, -nn.z};
    float s, u;
    seg_closest(q[0], q[1], q[2], q[3], &s, &u);
    float gap = dot(sub(seg_point(q[0], q[1], s), seg_point(q[2], q[3], u)), nn);
    if (!(gap - 2.0f * th < -1e-6f)) return false;
    float depth = (2.0f * th - gap) * 0.5f;
    float w[4] = {1.0f - s, s, 1.0f - u, u};
    float sa = w[0] * w[0] + w[1] * w[1], sb = w[2] * w[2] + w[3] * w[3];
    for (int k = 0; k < 4; k++) {
        float f = k < 2 ? (depth * w[k]) / sa : -((depth * w[k]) / sb);
        d[k] = V3{nn.x * f, nn.y * f, nn.z * f};
    }
    return true;
}

// ---------------------------------------------------------------------------
// response
// ---------------------------------------------------------------------------

// The side of the face that the vertex was on at the start of the step.
__device__ __forceinline__ bool vf_front(const V3* X) {
    V3 n0 = vnormalize(cross(sub(X[2], X[1]), sub(X[3], X[1])));
    return dot(sub(X[0], X[1]), n0) >= 0;
}

__device__ __forceinline__ bool vf_fix(bool front, const V3* q, float th, float min_n2, V3* d) {
    // VFResolveTest (CCD.cpp:1996-2032)
    V3 cr = cross(sub(q[2], q[1]), sub(q[3], q[1]));
    if (dot(cr, cr) <= min_n2) return false;
    V3 pn = vnormalize(cr);
    float s = front ? 1.0f : -1.0f;
    V3 sn = V3{pn.x * s, pn.y * s, pn.z * s};
    float depth0 = dot(sub(q[0], q[1]), sn) - 2.0 * th;
    if (!(depth0 < -1e-6)) return false;
    // VFResolveNew (CCD.cpp:2034-2090)
    V3 proj = V3{q[1].x + ((pn.x * s) * 2.0f) * th, q[1].y + ((pn.y * s) * 2.0f) * th, q[1].z + ((pn.z * s) * 2.0f) * th};
    float depth = dot(sub(proj, q[0]), sn) * 0.5;
    V3 wg = bary(q[0], q[1], q[2], q[3]);
    float sw = wg.x * wg.x + wg.y * wg.y + wg.z * wg.z;
    float wf[3] = {wg.x, wg.y, wg.z};
    float snv[3] = {sn.x, sn.y, sn.z}, pnv[3] = {pn.x, pn.y, pn.z};
    float qa[4][3] = {{q[0].x, q[0].y, q[0].z}, {q[1].x, q[1].y, q[1].z}, {q[2].x, q[2].y, q[2].z}, {q[3].x, q[3].y, q[3].z}};
    float fix[4][3];
    for (int a = 0; a < 3; a++) {
        float vfix = depth * snv[a];
        float ffix = depth * (pnv[a] * -s);
        fix[0][a] = (qa[0][a] + vfix) - qa[0][a];
        fix[1][a] = (qa[1][a] + (ffix * wf[0]) / sw) - qa[1][a];
        fix[2][a] = (qa[2][a] + (ffix * wf[1]) / sw) - qa[2][a];
        fix[3][a] = (qa[3][a] + (ffix * wf[2]) / sw) - qa[3][a];
    }
    for (int k = 0; k < 4; k++) d[k] = V3{fix[k][0], fix[k][1], fix[k][2]};
    return true;
}

// A contact's corners: vertex-face contacts (vertex, face) first, edge-edge
// ones (two edges) behind them.
__device__ __forceinline__ int4 contact_at(const int4* __restrict__ vquad, int nc, const int4* __restrict__ quad, int i) {
    return i < nc ? vquad[i] : quad[i - nc];
}
__device__ __forceinline__ int corner(int4 c, int k) { return k == 0 ? c.x : k == 1 ? c.y : k == 2 ? c.z : c.w; }

// The fix of corner k of a contact: doubled where the other side (face or
// vertex, or the other edge) is static as a whole.  `still`: bit per static corner.
__device__ __forceinline__ float fix_scale(bool vertex_face, unsigned still, int k) {
    if (vertex_face) return (k == 0 ? (still & 14) == 14 : (still & 1)) ? 2.0f : 1.0f;
    return (k < 2 ? (still & 12) == 12 : (still & 3) == 3) ? 2.0f : 1.0f;
}

__device__ __forceinline__ float mean_fix(unsigned long long sum, double c) {
    return (float)((double)(long long)sum / 4294967296.0 / c);
}

// The passes' sums of every vertex, and whether any has one.  A pass leaves p
// alone: the next one adds the means of the passes before to what it reads, and
// one launch at the end applies them all (a launch per pass less: 3000 contacts
// on 65,000 vertices, two passes: 18 us before, 12 so).
constexpr int RESOLVE_CHAIN = 4;
struct ResponseSums {
    unsigned long long* sum;  // [pass][vertex][3]
    int* count;               // [pass][vertex]
    int* touched;             // [vertex]
    int nv;
    // q moved by the first `passes` passes, as applying each in turn would
    __device__ __forceinline__ void move(float4& q, int v, int passes) const {
        int n[RESOLVE_CHAIN];
        unsigned long long s[RESOLVE_CHAIN][3];
#pragma unroll
        for (int j = 0; j < RESOLVE_CHAIN; j++)
            if (j < passes) {
                const size_t at = (size_t)j * nv + v;
                n[j] = count[at];
                for (int k = 0; k < 3; k++) s[j][k] = sum[3 * at + k];
            }
#pragma unroll
        for (int j = 0; j < RESOLVE_CHAIN; j++)
            if (j < passes && n[j]) {
                const double c = (double)n[j];
                q.x = q.x + mean_fix(s[j][0], c);
                q.y = q.y + mean_fix(s[j][1], c);
                q.z = q.z + mean_fix(s[j][2], c);
            }
    }
};

__global__ __launch_bounds__(256) void k_resolve_acc(const int4* __restrict__ vquad, int nc,
                                                     const int4* __restrict__ quad, int ne, const float4* __restrict__ x,
                                                     const float4* __restrict__ p, float th, float min_n2,
                                                     ResponseSums r, int pass) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nc + ne) return;
    const int4 c = contact_at(vquad, nc, quad, i);
    V3 X[4], q[4], d[4];
    unsigned still = 0;
    for (int k = 0; k < 4; k++) {
        float4 P = p[corner(c, k)];
        X[k] = v3(x[corner(c, k)]);
        r.move(P, corner(c, k), pass);
        q[k] = v3(P);
        if (P.w == 0.0f) still |= 1u << k;
    }
    if (!(i < nc ? vf_fix(vf_front(X), q, th, min_n2, d) : ee_fix(X, q, th, d))) return;
    for (int k = 0; k < 4; k++) {
        if (still >> k & 1) continue;
        const float sc = fix_scale(i < nc, still, k);
        const size_t at = (size_t)pass * r.nv + corner(c, k);
        atomicAdd(&r.sum[3 * at], (unsigned long long)to_fixed(d[k].x * sc));
        atomicAdd(&r.sum[3 * at + 1], (unsigned long long)to_fixed(d[k].y * sc));
        atomicAdd(&r.sum[3 * at + 2], (unsigned long long)to_fixed(d[k].z * sc));
        atomicAdd(&r.count[at], 1);
        r.touched[corner(c, k)] = 1;
    }
}

// Moves every vertex that a contact touched and clears its sums.  A vertex of
// several contacts is moved by the thread that takes its mark.
__global__ __launch_bounds__(256) void k_resolve_apply(const int4* __restrict__ vquad, int nc,
                                                       const int4* __restrict__ quad, int ne, ResponseSums r, int passes,
                                                       float4* __restrict__ p) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 4 * (nc + ne)) return;
    const int v = corner(contact_at(vquad, nc, quad, i >> 2), i & 3);
    if (!atomicExch(&r.touched[v], 0)) return;
    float4 q = p[v];
    r.move(q, v, passes);
    p[v] = q;
    for (int j = 0; j < passes; j++) {
        const size_t at = (size_t)j * r.nv + v;
        r.count[at] = 0;
        for (int k = 0; k < 3; k++) r.sum[3 * at + k] = 0;
    }
}

// Every pass of a few contacts in one workgroup, one contact per thread (350
// contacts, two passes: 8.4 us; three launches take 12, and with sums in global
// memory the workgroup took 30), with
// the touched vertices' positions and sums in an LDS table (open addressing by
// vertex id).  The contacts must have at most `slots` corners.
// The sums are integers, so this order gives the bits of any other.
constexpr int RESOLVE_BLOCK = 1024, RESOLVE_SLOTS = 3712, RESOLVE_SLOT_BYTES = 44;

__device__ __forceinline__ int resolve_slot(int* __restrict__ key, int slots, int v) {
    int s = (int)__umulhi((unsigned)v * 0x9E3779B1u, (unsigned)slots);
    for (;;) {  // ends: there are no more distinct vertices than slots
        const int old = atomicCAS(&key[s], -1, v);
        if (old == -1 || old == v) return s;
        s = s + 1 == slots ? 0 : s + 1;
    }
}

__global__ __launch_bounds__(RESOLVE_BLOCK) void k_resolve_few(const int4* __restrict__ vquad, int nc,
                                                               const int4* __restrict__ quad, int ne,
                                                               const float4* __restrict__ x, float4* __restrict__ p,
                                                               float th, float min_n2, int passes, int slots) {
    extern __shared__ unsigned long long lds_sums[];
    unsigned long long* sum = lds_sums;                       // 3 per slot
    float* at = reinterpret_cast<float*>(sum + 3 * slots);    // 3 per slot
    int* count = reinterpret_cast<int*>(at + 3 * slots);
    int* key = count + slots;
    const int i = threadIdx.x;
    const bool mine = i < nc + ne;
    const int4 c = mine ? contact_at(vquad, nc, quad, i) : make_int4(0, 0, 0, 0);
    for (int s = threadIdx.x; s < slots; s += blockDim.x) {
        sum[3 * s] = sum[3 * s + 1] = sum[3 * s + 2] = 0;
        count[s] = 0;
        key[s] = -1;
    }
    V3 X[4];
    float4 P[4];
    unsigned still = 0;
    if (mine)
        for (int k = 0; k < 4; k++) {
            P[k] = p[corner(c, k)];
            X[k] = v3(x[corner(c, k)]);
            if (P[k].w == 0.0f) still |= 1u << k;
        }
    __syncthreads();
    int slot[4] = {0, 0, 0, 0};
    bool front = false;
    if (mine) {
        front = vf_front(X);
        for (int k = 0; k < 4; k++) {
            slot[k] = resolve_slot(key, slots, corner(c, k));
            at[3 * slot[k]] = P[k].x;
            at[3 * slot[k] + 1] = P[k].y;
            at[3 * slot[k] + 2] = P[k].z;
        }
    }
    __syncthreads();
    for (int ps = 0; ps < passes; ps++) {
        V3 q[4], d[4];
        if (mine)
            for (int k = 0; k < 4; k++) q[k] = V3{at[3 * slot[k]], at[3 * slot[k] + 1], at[3 * slot[k] + 2]};
        if (mine && (i < nc ? vf_fix(front, q, th, min_n2, d) : ee_fix(X, q, th, d)))
            for (int k = 0; k < 4; k++) {
                if (still >> k & 1) continue;
                const float sc = fix_scale(i < nc, still, k);
                atomicAdd(&sum[3 * slot[k]], (unsigned long long)to_fixed(d[k].x * sc));
                atomicAdd(&sum[3 * slot[k] + 1], (unsigned long long)to_fixed(d[k].y * sc));
                atomicAdd(&sum[3 * slot[k] + 2], (unsigned long long)to_fixed(d[k].z * sc));
                atomicAdd(&count[slot[k]], 1);
            }
        __syncthreads();
        for (int s = threadIdx.x; s < slots; s += blockDim.x) {
            const int n = count[s];
            if (!n) continue;
            const double cn = (double)n;
            for (int a = 0; a < 3; a++) {
                at[3 * s + a] = at[3 * s + a] + mean_fix(sum[3 * s + a], cn);
                sum[3 * s + a] = 0;
            }
            count[s] = 0;
        }
        __syncthreads();
    }
    // w was not changed; a static vertex has no sum and its position is the one read
    for (int s = threadIdx.x; s < slots; s += blockDim.x) {
        const int v = key[s];
        if (v < 0) continue;
        p[v].x = at[3 * s];
        p[v].y = at[3 * s + 1];
        p[v].z = at[3 * s + 2];
    }
}

// ---------------------------------------------------------------------------
// host drivers
// ---------------------------------------------------------------------------
static inline int blocks(long long n) { return (int)((n + 255) / 256); }

// Working buffers only grow: detections of varying size reuse them instead
// of freeing and allocating (hipFree waits for the device) every time.
template <typename T>
static void grow(DBuf<T>& b, size_t n) {
    if (b.n < n || !b.ptr) b.alloc(std::max<size_t>(n, 1));
}

void Broadphase::build(hipStream_t s, const HashCfg& g, const float4* p, const int* tris, int nt) {
    cfg = g;
    this->nt = nt;
    grow(keys, std::max(1, nt));
    grow(ids, std::max(1, nt));
    grow(raw, std::max(1, nt));
    grow(k2, std::max(1, nt));
    grow(v2, std::max(1, nt));
    grow(hist, radix_hist_ints(nt));
    grow(cstart, std::max(1, g.ncells));
    grow(cend, std::max(1, g.ncells));
    build_sorted<false>(s, g, p, 0, tris, nt, keys.ptr, ids.ptr, raw.ptr, cstart.ptr, cend.ptr, k2.ptr, v2.ptr, hist.ptr);
}

void Broadphase::set_edges(hipStream_t s, const std::vector<int>& te, const std::vector<int2>& ed) {
    edge_tris = te.size() / 3;
    ehubs.forget();
    edges.upload(ed, s);
    nedges = (int)ed.size();
    // edge -> triangles (CSR)
    std::vector<int> eo(ed.size() + 1, 0), et(te.size());
    for (int e : te) eo[(size_t)e + 1]++;
    for (size_t e = 0; e < ed.size(); e++) eo[e + 1] += eo[e];
    std::vector<int> at(eo.begin(), eo.end() - 1);
    for (size_t i = 0; i < te.size(); i++) et[at[te[i]]++] = (int)(i / 3);
    etoff.upload(eo, s);
    etri.upload(et, s);
    // vertex -> neighbour CSR from the edges (each edge once, both directions)
    int nv = 0;
    for (const int2& e : ed) nv = std::max(nv, e.y + 1);
    std::vector<int> off((size_t)nv + 1, 0), nbr((size_t)2 * ed.size());
    for (const int2& e : ed) {
        off[e.x + 1]++;
        off[e.y + 1]++;
    }
    for (int v = 0; v < nv; v++) off[v + 1] += off[v];
    std::vector<int> fill(off.begin(), off.end() - 1);
    for (const int2& e : ed) {
        nbr[fill[e.x]++] = e.y;
        nbr[fill[e.y]++] = e.x;
    }
    for (int v = 0; v < nv; v++)
        if (off[v + 1] - off[v] > RING_SORTED) std::sort(nbr.begin() + off[v], nbr.begin() + off[v + 1]);
    voff.upload(off, s);
    vnbr.upload(nbr, s);
    PBD_HIP(hipStreamSynchronize(s));
}

// Vertex -> triangles of a triangle list.
void Broadphase::set_triangles(hipStream_t s, const int* tris, int nt_, int nv) {
    vhubs.forget();
    grow(vtoff, (size_t)nv + 1);
    grow(vtri, (size_t)3 * std::max(1, nt_));
    grow(cnt, (size_t)nv + 1);
    grow(scan_tmp, ((size_t)nv + 1) / SB + 2);
    PBD_HIP(hipMemsetAsync(cnt.ptr, 0, sizeof(int) * ((size_t)nv + 1), s));
    if (nt_ > 0) hipLaunchKernelGGL(k_vt_count, dim3(blocks(3ll * nt_)), dim3(256), 0, s, tris, 3 * nt_, cnt.ptr);
    device_scan(s, cnt.ptr, vtoff.ptr, nv + 1, scan_tmp.ptr);
    if (nt_ > 0)
        hipLaunchKernelGGL(k_vt_fill, dim3(blocks(3ll * nt_)), dim3(256), 0, s, tris, 3 * nt_, vtoff.ptr, cnt.ptr, vtri.ptr);
    PBD_HIP(hipGetLastError());
}

// Table sizes for n entries: at least one slot per entry.
static int table_bits_for(long long n) {
    int b = 10;
    while (b < 26 && (1ll << b) < n) b++;
    return b;
}

// The cleared table (slot counts after the counters, one fill for both).
void Broadphase::clear_table(hipStream_t s, int bits) {
    table_bits = bits;
    const size_t head = sizeof(DetectCounts) / sizeof(int);
    static_assert(sizeof(DetectCounts) % 16 == 0, "counters before the table");
    grow(table, head + (1ull << bits));
    grow(place, 1ull << bits);
    PBD_HIP(hipMemsetAsync(table.ptr, 0, sizeof(int) * (head + (1ull << bits)), s));
}
static DetectCounts* counts_of(const DBuf<int>& table) { return reinterpret_cast<DetectCounts*>(table.ptr); }
static int* slots_of(const DBuf<int>& table) { return table.ptr + sizeof(DetectCounts) / sizeof(int); }

// The counters as of this point of the stream.  Waits for them only, after it
// has queued what `meanwhile` queues (once), so that the GPU has work while the
// host reads.  Slot: 0 vertex-face, 1 edge-edge (one may be read inside the
// other's meanwhile).
DetectTotals Broadphase::read_counts(hipStream_t s, int slot, std::function<void()>* meanwhile) {
    if (!counts_h[slot]) {
        PBD_HIP(hipHostMalloc(&counts_h[slot], sizeof(DetectCounts), hipHostMallocDefault));
        PBD_HIP(hipEventCreateWithFlags(&counts_ready[slot], hipEventDisableTiming));
    }
    PBD_HIP(hipMemcpyAsync(counts_h[slot], table.ptr, sizeof(DetectCounts), hipMemcpyDeviceToHost, s));
    PBD_HIP(hipEventRecord(counts_ready[slot], s));
    if (meanwhile && *meanwhile) {
        std::function<void()> queue;
        queue.swap(*meanwhile);
        queue();
    }
    PBD_HIP(hipEventSynchronize(counts_ready[slot]));
    const DetectCounts& c = *static_cast<const DetectCounts*>(counts_h[slot]);
    DetectTotals t{0, 0, c.entries, 0, c.contacts, c.face_span, c.vertex_span, c.hubs};
    for (int b = 0; b < NEAR_BUCKETS; b++) {
        near_n[b] = c.bucket[b].near;
        t.pairs += c.bucket[b].pairs;
        t.near += near_n[b];
        t.near_most = std::max(t.near_most, near_n[b]);
    }
    return t;
}

// Room for n candidates per bucket of the list.
void Broadphase::grow_near(size_t n) { grow(near_, n * NEAR_BUCKETS); }
unsigned Broadphase::near_cap() const { return (unsigned)std::min<size_t>(near_.n / NEAR_BUCKETS, 0x7fffffff); }

// Workgroups of the candidate visits: each wave takes two vertices (edges) at
// a time, and enough waves to fill the GPU take them in turn.
static int visit_blocks(long long n) { return (int)std::max(1ll, std::min(2048ll, (n + 2 * VISIT_WAVES - 1) / (2 * VISIT_WAVES))); }

// The units of the hubs among n vertices (edges) with the CSR offsets off, asked
// for once per triangle list (edge table), when a visit has reported a hub.
void Broadphase::Hubs::find(hipStream_t s, const int* off, int n) {
    DBuf<unsigned long long> total;
    total.alloc(2);
    PBD_HIP(hipMemsetAsync(total.ptr, 0, 2 * sizeof(unsigned long long), s));
    hipLaunchKernelGGL(k_hub_count, dim3(blocks(n)), dim3(256), 0, s, off, n, total.ptr);
    PBD_HIP(hipGetLastError());
    unsigned long long u = 0;
    PBD_HIP(hipMemcpyAsync(&u, total.ptr, sizeof u, hipMemcpyDeviceToHost, s));
    PBD_HIP(hipStreamSynchronize(s));
    PBD_CHECK(u < (1ull << 26), PBD_ERR_LIMIT, "too many triangles around hubs");  // HUB_SLOTS * u in 32 bits
    grow(unit, (size_t)u);
    grow(set, (size_t)u * HUB_SLOTS);
    hipLaunchKernelGGL(k_hub_units, dim3(blocks(n)), dim3(256), 0, s, off, n, total.ptr + 1, unit.ptr);
    PBD_HIP(hipGetLastError());
    PBD_HIP(hipStreamSynchronize(s));  // `total` goes
    units = (int)u;
    known = true;
}

// Their sets at the triangles' current cells.
void Broadphase::Hubs::enter(hipStream_t s, const int* off, const int* tri, const int4* tcell) {
    PBD_HIP(hipMemsetAsync(set.ptr, 0xff, sizeof(int) * (size_t)units * HUB_SLOTS, s));
    hipLaunchKernelGGL(k_hub_enter, dim3(blocks(32ll * units)), dim3(256), 0, s, unit.ptr, units, off, tri, tcell, set.ptr);
    PBD_HIP(hipGetLastError());
}

// The visits of the vertices to the centroid-cell table.
void Broadphase::vf_candidates(hipStream_t s, const HashCfg& g, const float4* x, const float4* p, int nv, bool list,
                               unsigned cap) {
    const unsigned mask = (1u << table_bits) - 1;
    auto visit = [&](auto* k, int n) {
        hipLaunchKernelGGL(k, dim3(visit_blocks(n)), dim3(64 * VISIT_WAVES), 0, s, g, x, p, n, vtoff.ptr, vtri.ptr,
                           tcell.ptr, slots_of(table), place.ptr, mask, (const FaceRec*)rec.ptr, counts_of(table), near_.ptr,
                           cap, vhubs.unit.ptr, vhubs.set.ptr);
    };
    visit(list ? k_vf_candidates<true, false> : k_vf_candidates<false, false>, nv);
    if (vhubs.units > 0) {
        vhubs.enter(s, vtoff.ptr, vtri.ptr, tcell.ptr);
        visit(list ? k_vf_candidates<true, true> : k_vf_candidates<false, true>, vhubs.units);
    }
    PBD_HIP(hipGetLastError());
}

// The centroid-cell table of the faces at p.
void Broadphase::cells(hipStream_t s, const HashCfg& g, const float4* x, const float4* p, const int* tris, int nt_,
                       float th, bool culled) {
    cfg = g;
    nt = nt_;
    if (culled) grow(axes, (size_t)std::max(1, nt) * sizeof(FaceAxes));
    grow(tcell, std::max(1, nt));
    grow(raw_rank, std::max(1, nt));
    grow(rec, (size_t)std::max(1, nt) * sizeof(FaceRec));
    const int bits = table_bits_for(2ll * nt);
    clear_table(s, bits);
    const unsigned mask = (1u << table_bits) - 1;
    hipLaunchKernelGGL(k_face_cells, dim3(blocks(nt)), dim3(256), 0, s, g, p, tris, nt, mask, slots_of(table), tcell.ptr,
                       raw_rank.ptr);
    hipLaunchKernelGGL(k_slot_places<true>, dim3(((1 << table_bits) + PLACE_SLOTS - 1) / PLACE_SLOTS), dim3(256), 0, s,
                       (const int4*)slots_of(table), 1 << table_bits, (int4*)place.ptr, &counts_of(table)->entries);
    hipLaunchKernelGGL(k_cell_fill, dim3(blocks(nt)), dim3(256), 0, s, nt, tcell.ptr, raw_rank.ptr, slots_of(table),
                       place.ptr, x, p, tris, th, (FaceRec*)rec.ptr, culled ? (FaceAxes*)axes.ptr : nullptr);
    PBD_HIP(hipGetLastError());
}

void Broadphase::check_pairs(unsigned long long n, const char* what) {
    PBD_CHECK(n < (1ull << 31), PBD_ERR_LIMIT, std::string(what) + " overflows int32");
}

// Vertex-face contacts of one substep: candidates, narrowphase.  Lists that
// turn out too short are grown and the detection runs again.
void Broadphase::detect(hipStream_t s, const HashCfg& g, const HashCfg* swept, const float4* x, const float4* p,
                        const int* tris, int nt_, int nv, float th, bool store, std::function<void()> meanwhile) {
    npairs = ncontacts = 0;
    listed = false;
    cfg = g;
    nt = nt_;
    by_box = swept != nullptr;
    if (nt <= 0 || nv <= 0) {
        if (meanwhile) meanwhile();
        return;
    }
    grow_near(std::max<size_t>(1 << 10, (size_t)nv / NEAR_BUCKETS));
    grow_contacts(std::max<size_t>(1 << 14, (size_t)nv / 4), store);
    DetectTotals c{};
    for (;;) {
        const unsigned near_cap = this->near_cap(), cap = (unsigned)vquad.n;
        if (swept) {
            swept_table(s, g, *swept, x, p, tris, th);
            hipLaunchKernelGGL(k_swept_candidates, dim3(visit_blocks(nv)), dim3(64 * VISIT_WAVES), 0, s, g, *swept, x, p,
                               nv, vtoff.ptr, slots_of(table), place.ptr, (1u << table_bits) - 1, ent.ptr,
                               (unsigned)std::min<size_t>(ent.n, 0x7fffffff), (const FaceRec*)rec.ptr, sw_cell.ptr,
                               counts_of(table), near_.ptr, near_cap);
        } else {
            cells(s, g, x, p, tris, nt, th, true);
            vf_candidates(s, g, x, p, nv, false, near_cap);
        }
        auto* narrow = store ? k_narrow<true> : k_narrow<false>;
        hipLaunchKernelGGL(narrow, dim3(1024), dim3(256), 0, s, near_.ptr, near_cap, tris,
                           (const FaceAxes*)axes.ptr, x, p, th,
                           counts_of(table), cap, vquad.ptr, vf.ptr, rt.ptr, rn.ptr, rw.ptr);
        PBD_HIP(hipGetLastError());
        c = read_counts(s, 0, &meanwhile);
        if (c.hubs && !vhubs.known) {
            vhubs.find(s, vtoff.ptr, nv);
            continue;
        }
        if (swept) {
            PBD_CHECK(!c.face_span, PBD_ERR_LIMIT, "a face's swept box spans more than 4096 cells: use a larger cell");
            PBD_CHECK(c.entries < (1ull << 31), PBD_ERR_LIMIT, "swept-box cell entries overflow int32");
        }
        const bool table_short = swept && c.entries > ent.n;
        if (!table_short) {
            PBD_CHECK(!c.vertex_span, PBD_ERR_LIMIT,
                      "a vertex's swept box spans more than 4096 cells: use a larger cell");
            check_pairs(c.pairs, "candidate pair count");
        }
        if (!table_short && c.near_most <= near_cap && c.contacts <= cap) break;
        if (table_short) grow(ent, (size_t)c.entries + c.entries / 4);
        else if (c.near_most > near_cap) grow_near((size_t)c.near_most + c.near_most / 4);
        else grow_contacts((size_t)c.contacts + c.contacts / 4, store);
    }
    npairs = (long long)c.pairs;
    ncontacts = c.contacts;
    st_dets++;
    st_tris += nt;
    st_entries += swept ? (long long)c.entries : (long long)nt;
    st_raw += npairs;
    st_pairs += npairs;
    st_contacts += ncontacts;
    if (store) order_contacts(s, vf, nullptr, ncontacts, nv, ckey, nullptr);
}

void Broadphase::swept_table(hipStream_t s, const HashCfg& g, const HashCfg& gi, const float4* x, const float4* p,
                             const int* tris, float th) {
    grow(rec, (size_t)nt * sizeof(FaceRec));
    grow(axes, (size_t)nt * sizeof(FaceAxes));
    grow(sw_cell, 2 * (size_t)nt);
    grow(ent, 12 * (size_t)nt);
    clear_table(s, table_bits_for(2ll * nt));
    const unsigned mask = (1u << table_bits) - 1;
    hipLaunchKernelGGL(k_swept_faces, dim3(blocks(nt)), dim3(256), 0, s, g, gi, x, p, tris, nt, th, mask,
                       slots_of(table), sw_cell.ptr, (FaceRec*)rec.ptr, (FaceAxes*)axes.ptr, counts_of(table));
    hipLaunchKernelGGL(k_slot_places<false>, dim3(((1 << table_bits) + PLACE_SLOTS - 1) / PLACE_SLOTS), dim3(256), 0, s,
                       (const int4*)slots_of(table), 1 << table_bits, (int4*)place.ptr, &counts_of(table)->entries);
    hipLaunchKernelGGL(k_swept_fill, dim3(blocks((long long)FACE_LANES * nt)), dim3(256), 0, s, nt, sw_cell.ptr, mask, place.ptr,
                       ent.ptr, (unsigned)std::min<size_t>(ent.n, 0x7fffffff));
    PBD_HIP(hipGetLastError());
}

void Broadphase::grow_contacts(size_t n, bool store) {
    grow(vquad, n);
    if (!store) return;
    grow(vf, vquad.n);
    grow(rt, vquad.n);
    grow(rn, 3 * vquad.n);
    grow(rw, 4 * vquad.n);
}

// The n contacts of rt / rn / rw with ids `key` in ascending order of their
// ids, into okey (and oquad) / ct / cn / cw or their edge-edge counterparts.
void Broadphase::order_contacts(hipStream_t s, const DBuf<int2>& key, const int4* quad, long long n, int nfirst,
                                DBuf<int2>& okey, DBuf<int4>* oquad) {
    const size_t m = (size_t)std::max(1ll, n);
    DBuf<float>& ot = oquad ? ect : ct;
    DBuf<float>& on = oquad ? ecn : cn;
    DBuf<double>& ow = oquad ? ecw : cw;
    grow(okey, m);
    grow(ot, m);
    grow(on, 3 * m);
    grow(ow, 4 * m);
    if (oquad) grow(*oquad, m);
    if (n <= 0) return;
    grow(cnt, (size_t)nfirst + 1);
    grow(off, (size_t)nfirst + 1);
    grow(idx, m);
    grow(scan_tmp, ((size_t)nfirst + 1) / SB + 2);
    PBD_HIP(hipMemsetAsync(cnt.ptr, 0, sizeof(int) * ((size_t)nfirst + 1), s));
    hipLaunchKernelGGL(k_first_count, dim3(blocks(n)), dim3(256), 0, s, key.ptr, (int)n, cnt.ptr);
    device_scan(s, cnt.ptr, off.ptr, nfirst + 1, scan_tmp.ptr);
    hipLaunchKernelGGL(k_first_deal, dim3(blocks(n)), dim3(256), 0, s, key.ptr, (int)n, off.ptr, cnt.ptr, idx.ptr);
    hipLaunchKernelGGL(k_contact_order, dim3(blocks(n)), dim3(256), 0, s, key.ptr, (int)n, off.ptr, idx.ptr, rt.ptr,
                       rn.ptr, rw.ptr, quad, okey.ptr, ot.ptr, on.ptr, ow.ptr, oquad ? oquad->ptr : nullptr);
    PBD_HIP(hipGetLastError());
}

// Sorts the listed pairs by (first, second) into hi / lo.
void Broadphase::sort_near(hipStream_t s, int nfirst, int nsecond, DBuf<uint32_t>& hi, DBuf<uint32_t>& lo) {
    BucketPlaces b{};
    unsigned most = 0;
    for (int i = 0; i < NEAR_BUCKETS; i++) {
        b.at[i + 1] = b.at[i] + (int)near_n[i];
        most = std::max(most, near_n[i]);
    }
    const long long n = b.at[NEAR_BUCKETS];
    grow(hi, (size_t)std::max(1ll, n));
    grow(lo, (size_t)std::max(1ll, n));
    if (n <= 0) return;
    grow(k2, n);
    grow(v2, n);
    grow(hist, radix_hist_ints(n));
    hipLaunchKernelGGL(k_unzip, dim3(blocks(most), NEAR_BUCKETS), dim3(256), 0, s, near_.ptr, near_cap(), b, hi.ptr,
                       lo.ptr);
    int fb = 1, vb = 1;
    while (fb < 31 && (1ll << fb) < nsecond) fb++;
    while (vb < 31 && (1ll << vb) < nfirst) vb++;
    radix_sort_pairs(s, lo.ptr, hi.ptr, k2.ptr, v2.ptr, (int)n, fb, hist.ptr);
    radix_sort_pairs(s, hi.ptr, lo.ptr, k2.ptr, v2.ptr, (int)n, vb, hist.ptr);
}

// The centroid-cell candidates of the faces at p as sorted lists uv / uf.
long long Broadphase::list_pairs(hipStream_t s, const HashCfg& g, const float4* p, const int* tris, int nt_, int nv) {
    cfg = g;
    nt = nt_;
    npairs = 0;
    if (nt <= 0 || nv <= 0) return 0;
    if (!near_.n) grow_near(1 << 10);
    for (;;) {
        const unsigned cap = near_cap();
        cells(s, g, p, p, tris, nt, 0.0f, false);
        vf_candidates(s, g, p, p, nv, true, cap);
        const DetectTotals c = read_counts(s, 0, nullptr);
        if (c.hubs && !vhubs.known) {
            vhubs.find(s, vtoff.ptr, nv);
            continue;
        }
        check_pairs(c.near, "candidate pair count");
        npairs = (long long)c.near;
        if (c.near_most <= cap) break;
        grow_near(c.near_most);
    }
    sort_near(s, nv, nt, uv, uf);
    return npairs;
}

// The candidates of the last detect() as sorted lists uv / uf, made when first
// asked for.
void Broadphase::list_detected(hipStream_t s, const float4* p, const int* tris, int nv) {
    if (listed) return;
    const long long n = npairs;
    if (n > 0 && by_box) sort_near(s, nv, nt, uv, uf);
    else if (n > 0) list_pairs(s, cfg, p, tris, nt, nv);
    npairs = n;
    listed = true;
}

// The edge table of the faces' centroid cells at p, and its candidates.
void Broadphase::ee_candidates(hipStream_t s, const HashCfg& g, const float4* x, const float4* p, const int* tris,
                               int nt_, bool list, float th, unsigned cap) {
    cfg = g;
    nt = nt_;
    grow(tcell, std::max(1, nt));
    grow(rec, 3 * (size_t)std::max(1, nt) * sizeof(EdgeRec));
    clear_table(s, table_bits_for(2ll * nt));
    const unsigned mask = (1u << table_bits) - 1;
    EdgeRec* ent = reinterpret_cast<EdgeRec*>(rec.ptr);
    hipLaunchKernelGGL(k_tri_cells, dim3(blocks(nt)), dim3(256), 0, s, g, p, tris, nt, mask, tcell.ptr);
    hipLaunchKernelGGL(k_edge_count, dim3(blocks(nedges)), dim3(256), 0, s, nedges, etoff.ptr, etri.ptr, tcell.ptr,
                       slots_of(table));
    hipLaunchKernelGGL(k_slot_places<false>, dim3(((1 << table_bits) + PLACE_SLOTS - 1) / PLACE_SLOTS), dim3(256), 0, s,
                       (const int4*)slots_of(table), 1 << table_bits, (int4*)place.ptr, &counts_of(table)->entries);
    hipLaunchKernelGGL(k_edge_fill, dim3(blocks(nedges)), dim3(256), 0, s, nedges, edges.ptr, etoff.ptr, etri.ptr,
                       tcell.ptr, x, p, place.ptr, ent);
    auto visit = [&](auto* k, int n) {
        hipLaunchKernelGGL(k, dim3(visit_blocks(n)), dim3(64 * VISIT_WAVES), 0, s, g, n, edges.ptr, etoff.ptr,
                           etri.ptr, voff.ptr, vnbr.ptr, x, p, tcell.ptr, slots_of(table), place.ptr, mask, ent, th,
                           counts_of(table), near_.ptr, cap, ehubs.unit.ptr, ehubs.set.ptr);
    };
    visit(list ? k_ee_candidates<true, false> : k_ee_candidates<false, false>, nedges);
    if (ehubs.units > 0) {
        ehubs.enter(s, etoff.ptr, etri.ptr, tcell.ptr);
        visit(list ? k_ee_candidates<true, true> : k_ee_candidates<false, true>, ehubs.units);
    }
    PBD_HIP(hipGetLastError());
}

// Edge-edge contacts at p.
void Broadphase::detect_ee(hipStream_t s, const HashCfg& g, const float4* x, const float4* p, const int* tris, int nt_,
                           float th, bool store, std::function<void()> meanwhile) {
    ee_npairs = ee_ncontacts = 0;
    ee_listed = false;
    if (nt_ <= 0 || nedges <= 0) {
        if (meanwhile) meanwhile();
        return;
    }
    PBD_CHECK(edge_tris >= (size_t)nt_, PBD_ERR_STATE, "internal: edge table does not match the triangles");
    grow_near(std::max<size_t>(1 << 10, (size_t)nedges / NEAR_BUCKETS));
    auto grow_ee = [&](size_t n) {
        grow(quad, n);
        if (!store) return;
        grow(eab, quad.n);
        grow(rt, quad.n);
        grow(rn, 3 * quad.n);
        grow(rw, 4 * quad.n);
    };
    grow_ee(std::max<size_t>(1 << 14, (size_t)nedges / 8));
    DetectTotals c{};
    for (;;) {
        const unsigned near_cap = this->near_cap(), cap = (unsigned)quad.n;
        ee_candidates(s, g, x, p, tris, nt_, false, th, near_cap);
        auto* narrow = store ? k_narrow_ee<true> : k_narrow_ee<false>;
        hipLaunchKernelGGL(narrow, dim3(1024), dim3(256), 0, s, near_.ptr, near_cap, edges.ptr, x, p, th,
                           counts_of(table), cap, eab.ptr, quad.ptr, rt.ptr, rn.ptr, rw.ptr);
        PBD_HIP(hipGetLastError());
        c = read_counts(s, 1, &meanwhile);
        if (c.hubs && !ehubs.known) {
            ehubs.find(s, etoff.ptr, nedges);
            continue;
        }
        check_pairs(c.pairs, "edge-edge candidate count");
        if (c.near_most <= near_cap && c.contacts <= cap) break;
        if (c.near_most > near_cap) grow_near((size_t)c.near_most + c.near_most / 4);
        else grow_ee((size_t)c.contacts + c.contacts / 4);
    }
    ee_npairs = (long long)c.pairs;
    ee_ncontacts = c.contacts;
    st_ee_raw += ee_npairs;
    st_ee_pairs += ee_npairs;
    st_ee_contacts += ee_ncontacts;
    if (store) order_contacts(s, eab, quad.ptr, ee_ncontacts, nedges, eabs, &ecq);
}

// The edge-edge candidates of the last detect_ee() as sorted lists eua / eub.
void Broadphase::list_detected_ee(hipStream_t s, const HashCfg& g, const float4* x, const float4* p, const int* tris,
                                  float th) {
    if (ee_listed) return;
    if (ee_npairs > 0) {
        for (;;) {
            ee_candidates(s, g, x, p, tris, nt, true, th, near_cap());
            const DetectTotals c = read_counts(s, 0, nullptr);
            if (c.near_most <= near_cap()) break;
            grow_near(c.near_most);
        }
        sort_near(s, nedges, nedges, eua, eub);
    }
    ee_listed = true;
}

void Broadphase::resolve(hipStream_t s, const float4* x, float4* p, int nv, float th, int passes, float min_n2) {
    const int nc = (int)ncontacts, ne = (int)ee_ncontacts, n = nc + ne;
    if (n <= 0 || passes <= 0) return;
    st_resolved += (long long)n * passes;
    if (!few_slots) {
        // the LDS one workgroup may take on this device, asked for once
        few_slots = RESOLVE_SLOTS;
        if (hipFuncSetAttribute((const void*)k_resolve_few, hipFuncAttributeMaxDynamicSharedMemorySize,
                                RESOLVE_SLOTS * RESOLVE_SLOT_BYTES) != hipSuccess) {
            (void)hipGetLastError();  // the refusal is handled by the smaller limit
            few_slots = 65536 / RESOLVE_SLOT_BYTES;
        }
    }
    if (4 * n <= few_slots) {
        // Contacts of cloths share corners (a fifth of 4 n are distinct), others need not: a quarter more slots
        // than corners, as far as the LDS goes, keep the probes short there too (464 disjoint contacts, two passes:
        // 104 us with 4 n slots, 16 with 5 n; beyond 740 they fill the table, 87 us at 928 against 34 in chained
        // passes, which take 26 where corners are shared against 17 here).  The threads without a contact help
        // with the loops over the slots.
        const int slots = std::max(64, std::min(few_slots, 5 * n)), lds = slots * RESOLVE_SLOT_BYTES;
        const int threads = std::min(RESOLVE_BLOCK, (std::max(n, slots / 2) + 63) / 64 * 64);
        hipLaunchKernelGGL(k_resolve_few, dim3(1), dim3(threads), lds, s, vquad.ptr, nc, quad.ptr, ne, x, p,
                           th, min_n2, passes, slots);
        PBD_HIP(hipGetLastError());
        return;
    }
    const int chain = std::min(passes, RESOLVE_CHAIN);
    if (sums_nv != nv || sums_chain < chain) {
        // every response leaves them cleared
        sums_chain = std::max(sums_chain, chain);
        sums_nv = nv;
        grow(acc, (size_t)3 * sums_chain * nv);
        grow(vcnt, (size_t)(sums_chain + 1) * nv);
        PBD_HIP(hipMemsetAsync(acc.ptr, 0, sizeof(unsigned long long) * acc.n, s));
        PBD_HIP(hipMemsetAsync(vcnt.ptr, 0, sizeof(int) * vcnt.n, s));
    }
    const ResponseSums r{acc.ptr, vcnt.ptr + nv, vcnt.ptr, nv};
    for (int p0 = 0; p0 < passes; p0 += chain) {
        const int m = std::min(chain, passes - p0);
        for (int ps = 0; ps < m; ps++)
            hipLaunchKernelGGL(k_resolve_acc, dim3(blocks(n)), dim3(256), 0, s, vquad.ptr, nc, quad.ptr, ne, x,
                               (const float4*)p, th, min_n2, r, ps);
        hipLaunchKernelGGL(k_resolve_apply, dim3(blocks(4ll * n)), dim3(256), 0, s, vquad.ptr, nc, quad.ptr, ne, r, m, p);
    }
    PBD_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Broadphase build without allocation (pbd_sh_build_noalloc).  The caller
// brings device positions (3 floats per vertex), triangles and the output
// arrays; the radix sort runs in the caller's key and id arrays, with its
// ping-pong copies and digit counts in `scratch`, one static array per GPU
// that the process keeps until it ends.  Every call overwrites what it uses
// (digit counts and scans are written in full before they are read), so
// nothing carries over between calls; calls that overlap on one GPU race on
// it.
// ---------------------------------------------------------------------------
constexpr size_t SH_NOALLOC_HIST_INTS = (size_t)256 * (2 * (SH_NOALLOC_MAX_TRIS / RADIX_TILE) + 1);
constexpr size_t SH_NOALLOC_WORDS = 2 * (size_t)SH_NOALLOC_MAX_TRIS + SH_NOALLOC_HIST_INTS;
static __device__ __align__(256) uint32_t scratch[SH_NOALLOC_WORDS];

size_t sh_noalloc_scratch_bytes() { return sizeof(uint32_t) * SH_NOALLOC_WORDS; }

// Device address of this GPU's `scratch`, resolved once per device with the
// device current.  The host-side symbol is not a device address: only the
// resolved pointer is ever passed to a kernel.
static void* scratch_address(int device) {
    static std::mutex mu;
    static std::vector<void*> addr;
    std::lock_guard<std::mutex> lock(mu);
    if ((int)addr.size() <= device) addr.resize((size_t)device + 1, nullptr);
    if (!addr[device]) {
        void* p = nullptr;
        PBD_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        PBD_CHECK(p != nullptr, PBD_ERR_HIP, "hipGetSymbolAddress returned no address for the scratch array");
        addr[device] = p;
    }
    return addr[device];
}

void sh_build_noalloc(hipStream_t s, int device, const HashCfg& g, const float* pos, int nv, const int* tris, int nt,
                      int* sorted_keys, int* sorted_ids, int* raw_keys, int* cell_start, int* cell_end) {
    PBD_CHECK(nt <= SH_NOALLOC_MAX_TRIS, PBD_ERR_LIMIT,
              "pbd_sh_build_noalloc: " + std::to_string(nt) + " triangles exceed its maximum of " +
                  std::to_string(SH_NOALLOC_MAX_TRIS));
    uint32_t* scr = (uint32_t*)scratch_address(device);
    uint32_t* k2 = scr;
    uint32_t* v2 = scr + SH_NOALLOC_MAX_TRIS;
    int* hist = (int*)(scr + 2 * (size_t)SH_NOALLOC_MAX_TRIS);
    build_sorted<true>(s, g, pos, nv, tris, nt, (uint32_t*)sorted_keys, (uint32_t*)sorted_ids, raw_keys, cell_start,
                       cell_end, k2, v2, hist);
}

}  // namespace pbd
