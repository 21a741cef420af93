// bvh_gpu.hip -- a BVH built on the GPU (linear BVH), for scenes that must
// become resident fast (serving admission).  The reference builds its tree on
// the host (BVHAccelerator::new, bvh.rs:189-258, SAH); this builder makes a
// different tree over the same primitives, so a closest-hit query returns the
// reference's primitive, t and barycentrics except on rays where the
// reference's own answer depends on its visiting order: several primitives
// sharing the closest t (the later-visited one wins, bvh.rs:401-406 with
// mesh.rs:71), or a hit lying on its leaf box's rounded boundary, which the
// pop-time box test (bvh.rs:390-395) rejects once maxt has shrunk to that t
// and accepts before.  Occlusion bits are the reference's exactly (they do
// not depend on the tree).
//
// Pipeline, all on the device:
//   1. each primitive's box (the refined triple [c,b,a], mesh.rs:196-205;
//      spheres' boxes come from the host as build_bvh computes them) and
//      centroid (bvh.rs:77), the centroids' bounds, and the check that every
//      vertex index is in range;
//   2. 63-bit Morton codes (21 bits an axis);
//   3. radix sort of (code, prim) pairs (rocPRIM);
//   4. the binary radix tree over the sorted codes (T. Karras, "Maximizing
//      Parallelism in the Construction of BVHs, Octrees, and k-d Trees",
//      HPG 2012), duplicate codes split by their sorted position;
//   5. the sorted leaves' boxes and the boxes of aligned runs of 8, 64, 512 ..
//      of them; an interior node covers a run of leaves, so its box is the
//      union of a few of those;
//   6. depth-first positions in closed form (the reference layout: first child
//      at i + 1, second child at `off`);
//   7. the layouts the traversal kernels read: reference nodes, prim records
//      in leaf order, four-wide records (interior nodes at even depth, their
//      grandchildren as slots) and their compressed form.  Any-hit queries
//      walk the compressed records (there are no separate occlusion records).
// Nothing in it waits on another thread's result: steps 5 and 6 had been a
// climb with one atomic and two device-wide fences a node (1.84 ms of a
// 300,000-triangle build) and a launch a level (32 launches, 0.5 ms); they
// take 0.07 ms.  16.8M triangles, uploads included: 170 -> 36.5 ms.
#include <hip/hip_runtime.h>
#include <string.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <vector>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "../../include/pbrtx_gpu.h"
#include "bvh_build.hpp"
#include "capi_internal.hpp"

namespace px {
namespace {

constexpr int GB = 256;
constexpr uint32_t LEAF_BIT = 0x80000000u;  // child reference: a leaf (sorted position)
constexpr uint32_t LEFT_BIT = 0x80000000u;  // parent reference: from the first child
constexpr int MAX_LEVELS = 100;              // tree depth <= 63 code bits + 32 position bits + 1

struct DBox {
    float lo[3], hi[3];
};

// What the host reads back, written on the device.
struct Header {
    uint32_t nq;        // four-wide records
    uint32_t maxdepth;  // of the deepest leaf
    uint32_t bad_index; // a vertex index was out of range
    uint32_t bad_cq;    // a record that the compressed form cannot hold
    RNode root;
};

__device__ __forceinline__ float wave_min(float v) {
    for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o));
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}
// the block's bounds (lo, hi of thread 0 .. GB-1) to out[6], by its first wave
__device__ __forceinline__ void block_bounds(const float* lo, const float* hi, float* out) {
    __shared__ float s[6][GB / 64];
    const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
    for (int a = 0; a < 3; ++a) {
        const float l = wave_min(lo[a]), h = wave_max(hi[a]);
        if (lane == 0) { s[a][wid] = l; s[3 + a][wid] = h; }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        float v = s[threadIdx.x][0];
        for (uint32_t w = 1; w < GB / 64; ++w)
            v = threadIdx.x < 3 ? fminf(v, s[threadIdx.x][w]) : fmaxf(v, s[threadIdx.x][w]);
        out[threadIdx.x] = v;
    }
}

// 1. primitive boxes and centroids, and the bounds of each block's centroids.
// An index out of range is noted and read as the last vertex (the build then
// ends with an error).
__global__ __launch_bounds__(GB) void k_prim_boxes(const float* verts, uint32_t nverts, const uint32_t* idx,
                                                   uint32_t nfaces, const DBox* sph_box, uint32_t nsph, DBox* box,
                                                   float* cen, float* part, Header* hdr) {
    const uint32_t n = nfaces + nsph;
    float lo[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, hi[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    for (uint32_t i = blockIdx.x * GB + threadIdx.x; i < n; i += gridDim.x * GB) {
        DBox b;
        if (i < nfaces) {
            // Triangle::world_bound over [c, b, a] (mesh.rs:196-205): BBox::new
            // then unions (fmin / fmax, bbox.rs:155-168)
            b = DBox{{FLT_MAX, FLT_MAX, FLT_MAX}, {-FLT_MAX, -FLT_MAX, -FLT_MAX}};
            for (int k = 2; k >= 0; --k) {
                uint32_t vi = idx[3 * (size_t)i + k];
                if (vi >= nverts) {
                    hdr->bad_index = 1u;
                    vi = nverts - 1u;
                }
                const float* p = verts + 3 * (size_t)vi;
                for (int a = 0; a < 3; ++a) {
                    b.lo[a] = fminf(b.lo[a], p[a]);
                    b.hi[a] = fmaxf(b.hi[a], p[a]);
                }
            }
        } else {
            b = sph_box[i - nfaces];
        }
        box[i] = b;
        for (int a = 0; a < 3; ++a) {
            const float c = (b.lo[a] + b.hi[a]) * 0.5f;  // bvh.rs:77
            cen[3 * (size_t)i + a] = c;
            lo[a] = fminf(lo[a], c);
            hi[a] = fmaxf(hi[a], c);
        }
    }
    block_bounds(lo, hi, part + 6 * (size_t)blockIdx.x);
}
__global__ __launch_bounds__(GB) void k_cen_bounds(const float* part, uint32_t nb, float* out) {
    float lo[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, hi[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    for (uint32_t b = threadIdx.x; b < nb; b += GB)
        for (int a = 0; a < 3; ++a) {
            lo[a] = fminf(lo[a], part[6 * (size_t)b + a]);
            hi[a] = fmaxf(hi[a], part[6 * (size_t)b + 3 + a]);
        }
    block_bounds(lo, hi, out);
}

__device__ __forceinline__ uint64_t spread21(uint64_t v) {
    v &= 0x1FFFFFull;
    v = (v | (v << 32)) & 0x1F00000000FFFFull;
    v = (v | (v << 16)) & 0x1F0000FF0000FFull;
    v = (v | (v << 8)) & 0x100F00F00F00F00Full;
    v = (v | (v << 4)) & 0x10C30C30C30C30C3ull;
    v = (v | (v << 2)) & 0x1249249249249249ull;
    return v;
}
__global__ __launch_bounds__(GB) void k_morton(const float* cen, uint32_t n, const float* cb, uint64_t* key,
                                               uint32_t* val) {
    for (uint32_t i = blockIdx.x * GB + threadIdx.x; i < n; i += gridDim.x * GB) {
        uint64_t code = 0;
        for (int a = 0; a < 3; ++a) {
            const float ext = cb[3 + a] - cb[a];
            float u = ext > 0.0f ? (cen[3 * (size_t)i + a] - cb[a]) / ext : 0.0f;
            u = u == u ? fminf(fmaxf(u, 0.0f), 1.0f) : 0.0f;
            const uint64_t q = (uint64_t)fminf(u * 2097152.0f, 2097151.0f);
            code |= spread21(q) << (2 - a);
        }
        key[i] = code;
        val[i] = i;
    }
}

// 4. Karras' radix tree: internal node i (0 .. n-2) covers sorted positions
// [first, last]; its children are internal nodes or leaves (LEAF_BIT).
__device__ __forceinline__ int delta(const uint64_t* k, uint32_t n, int64_t i, int64_t j) {
    if (j < 0 || j >= (int64_t)n) return -1;
    const uint64_t x = k[i] ^ k[j];
    if (x) return __clzll((long long)x);
    return 64 + __clz((int)((uint32_t)i ^ (uint32_t)j));  // equal codes: by position
}
// parent[x] of an interior node: its parent, LEFT_BIT when it is the first child.
__global__ __launch_bounds__(GB) void k_karras(const uint64_t* k, uint32_t n, uint32_t* child, uint32_t* parent,
                                               uint2* range) {
    for (uint32_t ii = blockIdx.x * GB + threadIdx.x; ii + 1 < n; ii += gridDim.x * GB) {
        const int64_t i = ii;
        const int d = (delta(k, n, i, i + 1) - delta(k, n, i, i - 1)) >= 0 ? 1 : -1;
        const int dmin = delta(k, n, i, i - d);
        int64_t lmax = 2;
        while (delta(k, n, i, i + lmax * d) > dmin) lmax <<= 1;
        int64_t l = 0;
        for (int64_t t = lmax >> 1; t >= 1; t >>= 1)
            if (delta(k, n, i, i + (l + t) * d) > dmin) l += t;
        const int64_t j = i + l * d;
        const int dnode = delta(k, n, i, j);
        int64_t s = 0;
        for (int64_t t = (l + 1) >> 1;; t = (t + 1) >> 1) {
            if (delta(k, n, i, i + (s + t) * d) > dnode) s += t;
            if (t == 1) break;
        }
        const int64_t g = i + s * d + (d < 0 ? -1 : 0);
        const int64_t lo = i < j ? i : j, hi = i < j ? j : i;
        const uint32_t left = (lo == g) ? ((uint32_t)g | LEAF_BIT) : (uint32_t)g;
        const uint32_t right = (hi == g + 1) ? ((uint32_t)(g + 1) | LEAF_BIT) : (uint32_t)(g + 1);
        child[2 * ii] = left;
        child[2 * ii + 1] = right;
        range[ii] = make_uint2((uint32_t)lo, (uint32_t)hi);
        if (!(left & LEAF_BIT)) parent[left] = (uint32_t)ii | LEFT_BIT;
        if (!(right & LEAF_BIT)) parent[right] = (uint32_t)ii;
    }
}

__device__ __forceinline__ void grow(DBox& b, const DBox& c) {
    // Union<BBox> (bbox.rs:170-183); min and max give the same bits in any order
    for (int a = 0; a < 3; ++a) {
        b.lo[a] = fminf(b.lo[a], c.lo[a]);
        b.hi[a] = fmaxf(b.hi[a], c.hi[a]);
    }
}
__device__ __forceinline__ DBox empty_box() {
    return DBox{{FLT_MAX, FLT_MAX, FLT_MAX}, {-FLT_MAX, -FLT_MAX, -FLT_MAX}};
}

// 5a. Runs of boxes: level 0 holds the sorted leaves' boxes, level k the boxes
// of aligned runs of 8^k of them (the last run may be short).  One launch
// makes three levels from one: a block takes 512 boxes of level `base`, its
// 64 runs of 8, 8 runs of 64 and the run of 512.  val (level 0 only): where
// the sorted leaves' boxes are.  Streaming: 24 B in and 27 out a leaf.
constexpr int RUN_LEVELS = 11;  // 8^10 = 2^30 leaves
struct Runs {
    DBox* box;
    uint32_t first[RUN_LEVELS], count[RUN_LEVELS];  // a level's boxes: box[first ..]
    uint32_t levels;
};
constexpr int RUN_B = 512;
__global__ __launch_bounds__(RUN_B) void k_runs(Runs r, uint32_t base, const uint32_t* val, const DBox* pbox) {
    __shared__ DBox s0[RUN_B], s1[RUN_B / 8], s2[RUN_B / 64];
    const uint32_t t = threadIdx.x, i = blockIdx.x * RUN_B + t;
    DBox b = empty_box();
    if (i < r.count[base]) {
        if (val) {
            b = pbox[val[i]];
            r.box[r.first[base] + i] = b;
        } else {
            b = r.box[r.first[base] + i];
        }
    }
    s0[t] = b;
    __syncthreads();
    if (t < RUN_B / 8 && base + 1 < r.levels) {
        DBox c = empty_box();
        for (int k = 0; k < 8; ++k) grow(c, s0[8 * t + k]);
        s1[t] = c;
        const uint32_t j = blockIdx.x * (RUN_B / 8) + t;
        if (j < r.count[base + 1]) r.box[r.first[base + 1] + j] = c;
    }
    __syncthreads();
    if (t < RUN_B / 64 && base + 2 < r.levels) {
        DBox c = empty_box();
        for (int k = 0; k < 8; ++k) grow(c, s1[8 * t + k]);
        s2[t] = c;
        const uint32_t j = blockIdx.x * (RUN_B / 64) + t;
        if (j < r.count[base + 2]) r.box[r.first[base + 2] + j] = c;
    }
    __syncthreads();
    if (t == 0 && base + 3 < r.levels) {
        DBox c = empty_box();
        for (int k = 0; k < 8; ++k) grow(c, s2[k]);
        r.box[r.first[base + 3] + blockIdx.x] = c;
    }
}

// 5b, 6. An interior node's box from its leaves lo .. hi: level by level the
// boxes up to the next aligned run from either end, then whole runs (half the
// nodes hold two leaves; a node of m leaves reads at most 14 log8 m boxes).
// Its depth-first position: before it come its ancestors and, for each of
// them that it lies in the second child of, the whole first child, 2m - 1
// nodes for m leaves; those leaves are the lo before its own, so the position
// is 2 lo + the ancestors that it lies in the first child of.  A leaf's is the
// same.
__global__ __launch_bounds__(GB) void k_nodes(uint32_t n, const uint32_t* child, const uint32_t* parent,
                                              const uint2* range, Runs r, DBox* ibox, uint32_t* pos_i,
                                              uint32_t* pos_l, uint32_t* depth_i, Header* hdr) {
    uint32_t deepest = 0, recs = 0;
    for (uint32_t x = blockIdx.x * GB + threadIdx.x; x + 1 < n; x += gridDim.x * GB) {
        const uint2 rg = range[x];
        uint32_t lo = rg.x, hi = rg.y;
        const uint32_t first = lo;
        DBox b = empty_box();
        // a run's box may be joined twice, so the ends take seven boxes each,
        // whatever lies before the next aligned run: independent loads
        for (uint32_t lv = 0;; ++lv) {
            const DBox* box = r.box + r.first[lv];
            if (hi - lo < 16u) {
                for (uint32_t k = 0; k <= hi - lo; k += 4)
#pragma unroll
                    for (uint32_t u = 0; u < 4; ++u) grow(b, box[min(lo + k + u, hi)]);
                break;
            }
#pragma unroll
            for (uint32_t k = 0; k < 7; ++k) {
                grow(b, box[lo + k]);
                grow(b, box[hi - k]);
            }
            lo = (lo + 7u) >> 3;
            hi = ((hi + 1u) >> 3) - 1u;
        }
        ibox[x] = b;
        uint32_t depth = 0, lefts = 0;
        for (uint32_t y = x; y != 0u;) {
            const uint32_t p = parent[y];
            ++depth;
            lefts += p >> 31;
            y = p & ~LEFT_BIT;
        }
        pos_i[x] = 2u * first + lefts;
        depth_i[x] = depth;
        deepest = max(deepest, depth + 1u);
        recs += (depth & 1u) ^ 1u;  // a record starts at every even depth
        const uint32_t L = child[2 * x], R = child[2 * x + 1];
        if (L & LEAF_BIT) pos_l[L & ~LEAF_BIT] = 2u * (L & ~LEAF_BIT) + lefts + 1u;
        if (R & LEAF_BIT) pos_l[R & ~LEAF_BIT] = 2u * (R & ~LEAF_BIT) + lefts;
    }
    __shared__ uint32_t s_deep, s_recs;
    if (threadIdx.x == 0) s_deep = s_recs = 0u;
    __syncthreads();
    atomicMax(&s_deep, deepest);
    atomicAdd(&s_recs, recs);
    __syncthreads();
    if (threadIdx.x == 0 && s_deep) {
        atomicMax(&hdr->maxdepth, s_deep);
        atomicAdd(&hdr->nq, s_recs);
    }
}

// 7a. reference nodes in depth-first order, record flags, prim records
__global__ __launch_bounds__(GB) void k_rnodes(uint32_t n, const uint32_t* child, const DBox* ibox, const DBox* leaf,
                                               const uint32_t* pos_i, const uint32_t* pos_l, const uint32_t* depth_i,
                                               RNode* rn, uint32_t* is_rec) {
    const uint32_t total = 2 * n - 1;
    for (uint32_t t = blockIdx.x * GB + threadIdx.x; t < total; t += gridDim.x * GB) {
        if (t < n - 1) {
            // interior node t: the children's axis of greatest centre separation
            // picks the near child (bvh.rs:409-415 reads the node's axis)
            const uint32_t L = child[2 * t], R = child[2 * t + 1];
            const DBox bl = (L & LEAF_BIT) ? leaf[L & ~LEAF_BIT] : ibox[L];
            const DBox br = (R & LEAF_BIT) ? leaf[R & ~LEAF_BIT] : ibox[R];
            int axis = 0;
            float best = -1.0f;
            for (int a = 0; a < 3; ++a) {
                const float sep = fabsf((br.lo[a] + br.hi[a]) - (bl.lo[a] + bl.hi[a]));
                if (sep > best) { best = sep; axis = a; }
            }
            RNode r;
            const DBox& b = ibox[t];
            for (int a = 0; a < 3; ++a) { r.lo[a] = b.lo[a]; r.hi[a] = b.hi[a]; }
            r.off = (R & LEAF_BIT) ? pos_l[R & ~LEAF_BIT] : pos_i[R];
            r.meta = (uint32_t)axis;
            rn[pos_i[t]] = r;
            is_rec[pos_i[t]] = (depth_i[t] & 1u) == 0u ? 1u : 0u;
        } else {
            const uint32_t j = t - (n - 1);  // leaf at sorted position j
            RNode r;
            const DBox& b = leaf[j];
            for (int a = 0; a < 3; ++a) { r.lo[a] = b.lo[a]; r.hi[a] = b.hi[a]; }
            r.off = j;
            r.meta = 3u | (1u << 2);
            const uint32_t p = n == 1 ? 0u : pos_l[j];
            rn[p] = r;
            is_rec[p] = 0u;
        }
    }
}

__device__ __forceinline__ float as_f(uint32_t u) { return __uint_as_float(u); }

__global__ __launch_bounds__(GB) void k_prim_recs(uint32_t n, uint32_t nfaces, const uint32_t* val,
                                                  const float* verts, uint32_t nverts, const uint32_t* idx,
                                                  const DBox* leaf, PrimRec* pr, PrimRec64* pr64, uint32_t* order) {
    for (uint32_t j = blockIdx.x * GB + threadIdx.x; j < n; j += gridDim.x * GB) {
        const uint32_t id = val[j];
        order[j] = id;
        PrimRec r;
        for (int k = 0; k < 12; ++k) r.w[k] = 0.0f;
        r.w[10] = as_f(id);
        uint32_t kind;
        if (id < nfaces) {
            // (an index out of range is the last vertex, as in k_prim_boxes)
            const float* p1 = verts + 3 * (size_t)min(idx[3 * (size_t)id + 2], nverts - 1u);
            const float* p2 = verts + 3 * (size_t)min(idx[3 * (size_t)id + 1], nverts - 1u);
            const float* p3 = verts + 3 * (size_t)min(idx[3 * (size_t)id + 0], nverts - 1u);
            for (int a = 0; a < 3; ++a) {
                r.w[a] = p1[a];
                r.w[3 + a] = p2[a] - p1[a];
                r.w[6 + a] = p3[a] - p1[a];
            }
            kind = 0u;
        } else {
            r.w[9] = as_f(id - nfaces);
            kind = 1u;
        }
        kind |= 0x100u;  // one prim a leaf: every record is its leaf's last
        r.w[11] = as_f(kind);
        pr[j] = r;
        // the 64-byte record: the leaf's exact box beside the triangle
        PrimRec64 q;
        for (int k = 0; k < 9; ++k) q.w[k] = r.w[k];
        if ((kind & 0xFFu) != 0u) q.w[0] = r.w[9];
        const DBox b = leaf[j];
        for (int a = 0; a < 3; ++a) { q.w[9 + a] = b.lo[a]; q.w[12 + a] = b.hi[a]; }
        q.w[15] = r.w[11];
        pr64[j] = q;
    }
}

// 7b. four-wide records: record q at depth-first position a (an interior
// node at even depth), slots = the grandchildren through each child (a leaf
// child is a slot itself); refs: ~(prim position) for a leaf, else the
// record index of the node (qidx = exclusive scan of is_rec)
__device__ __forceinline__ bool is_leaf_node(const RNode& r) { return (r.meta & 3u) == 3u; }
// rec[q] = the position of record q; and the root for the host
__global__ __launch_bounds__(GB) void k_rec_list(uint32_t nnodes, const uint32_t* is_rec, const uint32_t* qidx,
                                                 const RNode* rn, uint32_t* rec, Header* hdr) {
    for (uint32_t a = blockIdx.x * GB + threadIdx.x; a < nnodes; a += gridDim.x * GB) {
        if (is_rec[a]) rec[qidx[a]] = a;
        if (a == 0) hdr->root = rn[0];
    }
}
// 7c. the compressed records (as compress_records on the host: per axis the
// smallest power-of-two scale that spans the union box in 255 steps, bytes
// rounded outward and checked against the float the traversal decodes)
__device__ __forceinline__ float cq_decode_d(float o, uint32_t q, float s) {
    const float t = (float)q * s;  // exact
    return o + t;
}
__device__ bool cq_axis_d(float ulo, float uhi, const float* lo, const float* hi, const bool* used, uint8_t* qlo,
                          uint8_t* qhi, uint32_t* ebyte) {
    if (!(fabsf(ulo) <= FLT_MAX) || !(fabsf(uhi) <= FLT_MAX)) return false;
    const double ext = (double)uhi - (double)ulo;
    int e = -126;
    if (ext > 0.0) {
        e = (int)ceil(log2(ext / 255.0));
        if (e < -126) e = -126;
    }
    for (;; ++e) {
        if (e > 119) return false;
        if (cq_decode_d(ulo, 255u, ldexpf(1.0f, e)) >= uhi) break;
    }
    const float s = ldexpf(1.0f, e);
    for (int k = 0; k < 4; ++k) {
        if (!used[k]) { qlo[k] = 255; qhi[k] = 0; continue; }
        const double a = floor(((double)lo[k] - (double)ulo) / (double)s);
        int ql = a < 0 ? 0 : (a > 255 ? 255 : (int)a);
        while (ql > 0 && cq_decode_d(ulo, (uint32_t)ql, s) > lo[k]) --ql;
        const double b = ceil(((double)hi[k] - (double)ulo) / (double)s);
        int qh = b < 0 ? 0 : (b > 255 ? 255 : (int)b);
        while (qh < 255 && cq_decode_d(ulo, (uint32_t)qh, s) < hi[k]) ++qh;
        if (cq_decode_d(ulo, (uint32_t)ql, s) > lo[k] || cq_decode_d(ulo, (uint32_t)qh, s) < hi[k]) return false;
        qlo[k] = (uint8_t)ql;
        qhi[k] = (uint8_t)qh;
    }
    *ebyte = (uint32_t)(e + 127);
    return true;
}
__global__ __launch_bounds__(GB) void k_records(uint32_t nq, const uint32_t* rec, const RNode* rn,
                                                const uint32_t* qidx, QNode* qn, CNode* cn, Header* hdr) {
    for (uint32_t i = blockIdx.x * GB + threadIdx.x; i < nq; i += gridDim.x * GB) {
        const uint32_t a = rec[i];
        QNode q;
        const uint32_t b = a + 1, c = rn[a].off;
        uint32_t s[4];
        const uint32_t none = 0xFFFFFFFFu;
        if (is_leaf_node(rn[b])) { s[0] = b; s[1] = none; } else { s[0] = b + 1; s[1] = rn[b].off; }
        if (is_leaf_node(rn[c])) { s[2] = c; s[3] = none; } else { s[2] = c + 1; s[3] = rn[c].off; }
        const uint32_t ab = is_leaf_node(rn[b]) ? 0u : (rn[b].meta & 3u);
        const uint32_t ac = is_leaf_node(rn[c]) ? 0u : (rn[c].meta & 3u);
        q.meta = (rn[a].meta & 3u) | (ab << 2) | (ac << 4);
        q.pad[0] = q.pad[1] = q.pad[2] = 0u;
        for (int k = 0; k < 4; ++k) {
            if (s[k] == none) {
                q.ref[k] = QEMPTY;
                q.lx[k] = q.ly[k] = q.lz[k] = FLT_MAX;
                q.hx[k] = q.hy[k] = q.hz[k] = -FLT_MAX;
                continue;
            }
            const RNode& r = rn[s[k]];
            q.ref[k] = is_leaf_node(r) ? ~(int32_t)r.off : (int32_t)qidx[s[k]];
            q.lx[k] = r.lo[0]; q.ly[k] = r.lo[1]; q.lz[k] = r.lo[2];
            q.hx[k] = r.hi[0]; q.hy[k] = r.hi[1]; q.hz[k] = r.hi[2];
        }
        qn[i] = q;
        CNode cr;
        bool used[4];
        float u[6] = {FLT_MAX, FLT_MAX, FLT_MAX, -FLT_MAX, -FLT_MAX, -FLT_MAX};
        for (int k = 0; k < 4; ++k) {
            used[k] = q.ref[k] != QEMPTY;
            cr.ref[k] = q.ref[k];
            if (!used[k]) continue;
            u[0] = fminf(u[0], q.lx[k]); u[1] = fminf(u[1], q.ly[k]); u[2] = fminf(u[2], q.lz[k]);
            u[3] = fmaxf(u[3], q.hx[k]); u[4] = fmaxf(u[4], q.hy[k]); u[5] = fmaxf(u[5], q.hz[k]);
        }
        uint32_t ex = 0, ey = 0, ez = 0;
        if (!cq_axis_d(u[0], u[3], q.lx, q.hx, used, cr.q + 0, cr.q + 4, &ex) ||
            !cq_axis_d(u[1], u[4], q.ly, q.hy, used, cr.q + 8, cr.q + 12, &ey) ||
            !cq_axis_d(u[2], u[5], q.lz, q.hz, used, cr.q + 16, cr.q + 20, &ez)) {
            hdr->bad_cq = 1u;
            continue;
        }
        cr.ox = u[0]; cr.oy = u[1]; cr.oz = u[2];
        cr.emeta = ex | (ey << 8) | (ez << 16) | ((q.meta & 63u) << 24);
        cr.pad[0] = cr.pad[1] = 0u;
        cn[i] = cr;
    }
}

uint32_t grid_for(uint64_t n) {
    const uint64_t b = (n + GB - 1) / GB;
    return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(b, (uint64_t)device_cu_count() * 16));
}

// One device allocation for several arrays: take() them all twice, before
// alloc() to add up their bytes and after it to have their places.
struct Slab {
    uint8_t* p = nullptr;
    size_t at = 0;
    ~Slab() {
        if (p) (void)hipFree(p);
    }
    template <typename U>
    void take(U** out, size_t count) {
        *out = reinterpret_cast<U*>(p + at);
        at += (std::max<size_t>(count, 1) * sizeof(U) + 255) / 256 * 256;
    }
    hipError_t alloc() {
        const hipError_t e = hipMalloc((void**)&p, at);
        at = 0;
        return e;
    }
    void* release() {
        void* q = p;
        p = nullptr;
        return q;
    }
};

#define GCHK(x)                                          \
    do {                                                 \
        hipError_t e_ = (x);                             \
        if (e_ != hipSuccess) return hip_fail(e_, #x);   \
    } while (0)

}  // namespace

// The spheres' world boxes and records, as build_bvh makes them (host; a
// handful per scene).
static bool sphere_inputs(const SphereIn* sph, uint32_t nsph, std::vector<DBox>* boxes,
                          std::vector<SphereRec>* recs, std::string* err) {
    // reuse the host builder's exact per-sphere arithmetic: build a one-sphere
    // tree and take its record and root box
    boxes->resize(nsph);
    recs->resize(nsph);
    for (uint32_t s = 0; s < nsph; ++s) {
        HostBvh h;
        if (!build_bvh(nullptr, 0, nullptr, 0, sph + s, 1, 0, 1, &h, err)) return false;
        (*recs)[s] = h.spheres[0];
        for (int a = 0; a < 3; ++a) { (*boxes)[s].lo[a] = h.root_lo[a]; (*boxes)[s].hi[a] = h.root_hi[a]; }
    }
    return true;
}

int gpu_build_scene(const float* verts, uint32_t nverts, const uint32_t* idx, uint32_t nfaces, const SphereIn* sph,
                    uint32_t nsph, DeviceScene* S, double* build_ms) {
    auto t0 = std::chrono::steady_clock::now();
    memset(S, 0, sizeof(*S));
    const uint64_t N64 = (uint64_t)nfaces + nsph;
    if (N64 == 0) return fail(PBRTX_ERR_BUILD, "scene has no primitives");
    if (N64 >= (1ull << 30)) return fail(PBRTX_ERR_BUILD, "too many primitives");
    if (nfaces && (!verts || !idx)) return fail(PBRTX_ERR_ARG, "null mesh arrays");
    if (nsph && !sph) return fail(PBRTX_ERR_ARG, "null sphere array");
    if (nfaces && nverts == 0) return fail(PBRTX_ERR_BUILD, "vertex index out of range");
    std::string err;
    std::vector<DBox> sbox;
    std::vector<SphereRec> srec;
    if (!sphere_inputs(sph, nsph, &sbox, &srec, &err)) return fail(PBRTX_ERR_BUILD, err);
    const uint32_t n = (uint32_t)N64;
    const uint32_t nnodes = 2 * n - 1;
    hipStream_t st = nullptr;
    // the boxes' runs: level k holds ceil(n / 8^k)
    Runs runs{};
    uint32_t nruns = 0;
    for (uint64_t c = n;; c = (c + 7) / 8) {
        runs.first[runs.levels] = nruns;
        runs.count[runs.levels++] = (uint32_t)c;
        nruns += (uint32_t)c;
        if (c == 1) break;
    }
    const uint32_t nb = grid_for(n);
    size_t sort_bytes = 0, scan_bytes = 0;
    GCHK(rocprim::radix_sort_pairs((void*)nullptr, sort_bytes, (uint64_t*)nullptr, (uint64_t*)nullptr,
                                   (uint32_t*)nullptr, (uint32_t*)nullptr, n, 0, 63, st));
    GCHK(rocprim::exclusive_scan((void*)nullptr, scan_bytes, (uint32_t*)nullptr, (uint32_t*)nullptr, 0u, nnodes,
                                 rocprim::plus<uint32_t>(), st));
    // One allocation holds everything that the build itself needs and one the
    // scene: an allocation costs some 0.1 ms, a release 0.1-0.2 and a wait for
    // the device (40 of each: 4 of the 7.5 ms of a 300,000-triangle build).
    float *d_verts, *d_cen, *d_part, *d_cb;
    uint32_t *d_idx, *d_val, *d_val2, *d_child, *d_parent, *d_posi, *d_posl, *d_depth, *d_isrec, *d_qidx;
    uint64_t *d_key, *d_key2;
    uint2* d_range;
    DBox *d_pbox, *d_sbox, *d_ibox;
    Header* d_hdr;
    uint8_t *sort_tmp, *scan_tmp;
    Slab T;
    for (int pass = 0; pass < 2; ++pass) {
        T.take(&d_verts, 3 * (size_t)nverts);
        T.take(&d_idx, 3 * (size_t)nfaces);
        T.take(&d_sbox, nsph);
        T.take(&d_pbox, n);
        T.take(&d_cen, 3 * (size_t)n);
        T.take(&d_part, 6 * (size_t)nb);
        T.take(&d_cb, 6);
        T.take(&d_key, n);
        T.take(&d_key2, n);
        T.take(&d_val, n);
        T.take(&d_val2, n);
        T.take(&sort_tmp, sort_bytes);
        T.take(&scan_tmp, scan_bytes);
        T.take(&d_child, 2 * (size_t)n);
        T.take(&d_parent, n);
        T.take(&d_range, n);
        T.take(&runs.box, nruns);
        T.take(&d_ibox, n);
        T.take(&d_posi, n);
        T.take(&d_posl, n);
        T.take(&d_depth, n);
        T.take(&d_isrec, nnodes);
        T.take(&d_qidx, nnodes);
        T.take(&d_hdr, 1);
        if (pass == 0) GCHK(T.alloc());
    }
    GCHK(fill_u32((uint32_t*)d_hdr, 0u, sizeof(Header) / 4, st));
    if (nverts) GCHK(hipMemcpyAsync(d_verts, verts, 12 * (size_t)nverts, hipMemcpyHostToDevice, st));
    if (nfaces) GCHK(hipMemcpyAsync(d_idx, idx, 12 * (size_t)nfaces, hipMemcpyHostToDevice, st));
    if (nsph) GCHK(hipMemcpyAsync(d_sbox, sbox.data(), sizeof(DBox) * nsph, hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(k_prim_boxes, dim3(nb), dim3(GB), 0, st, d_verts, nverts, d_idx, nfaces, d_sbox, nsph, d_pbox,
                       d_cen, d_part, d_hdr);
    hipLaunchKernelGGL(k_cen_bounds, dim3(1), dim3(GB), 0, st, d_part, nb, d_cb);
    hipLaunchKernelGGL(k_morton, dim3(grid_for(n)), dim3(GB), 0, st, d_cen, n, d_cb, d_key, d_val);
    GCHK(hipGetLastError());
    GCHK(rocprim::radix_sort_pairs((void*)sort_tmp, sort_bytes, d_key, d_key2, d_val, d_val2, n, 0, 63, st));
    std::swap(d_key, d_key2);
    std::swap(d_val, d_val2);
    if (n > 1) {
        hipLaunchKernelGGL(k_karras, dim3(grid_for(n)), dim3(GB), 0, st, d_key, n, d_child, d_parent, d_range);
        GCHK(hipGetLastError());
    }
    for (uint32_t lv = 0; lv == 0 || lv + 1 < runs.levels; lv += 3)
        hipLaunchKernelGGL(k_runs, dim3((runs.count[lv] + RUN_B - 1) / RUN_B), dim3(RUN_B), 0, st, runs, lv,
                           lv == 0 ? d_val : (const uint32_t*)nullptr, d_pbox);
    GCHK(hipGetLastError());
    if (n > 1) {
        hipLaunchKernelGGL(k_nodes, dim3(grid_for(n)), dim3(GB), 0, st, n, d_child, d_parent, d_range, runs, d_ibox,
                           d_posi, d_posl, d_depth, d_hdr);
        GCHK(hipGetLastError());
    }
    Header hdr;
    GCHK(hipMemcpyAsync(&hdr, d_hdr, sizeof(hdr), hipMemcpyDeviceToHost, st));
    GCHK(hipStreamSynchronize(st));
    if (hdr.bad_index) return fail(PBRTX_ERR_BUILD, "vertex index out of range");
    const uint32_t nq = hdr.nq, maxd = hdr.maxdepth;
    if (n > 1 && maxd + 1 >= (uint32_t)MAX_LEVELS) return fail(PBRTX_ERR_BUILD, "linear BVH deeper than expected");
    // layouts
    RNode* d_rn;
    PrimRec* d_pr;
    PrimRec64* d_pr64;
    uint32_t* d_order;
    SphereRec* d_s;
    QNode* d_qn;
    CNode* d_cn;
    Slab A;
    for (int pass = 0; pass < 2; ++pass) {
        A.take(&d_rn, nnodes);
        A.take(&d_pr, n);
        A.take(&d_pr64, n);
        A.take(&d_order, n);
        A.take(&d_s, nsph);
        A.take(&d_qn, nq);
        A.take(&d_cn, nq);
        if (pass == 0) GCHK(A.alloc());
    }
    S->d_rnodes = A.release();  // holds the other arrays as well
    hipLaunchKernelGGL(k_rnodes, dim3(grid_for(nnodes)), dim3(GB), 0, st, n, d_child, d_ibox, runs.box, d_posi, d_posl,
                       d_depth, d_rn, d_isrec);
    hipLaunchKernelGGL(k_prim_recs, dim3(grid_for(n)), dim3(GB), 0, st, n, nfaces, d_val, d_verts, nverts, d_idx,
                       runs.box, d_pr, d_pr64, d_order);
    GCHK(hipGetLastError());
    GCHK(rocprim::exclusive_scan((void*)scan_tmp, scan_bytes, d_isrec, d_qidx, 0u, nnodes, rocprim::plus<uint32_t>(),
                                 st));
    // (the list takes the place of the interior nodes' positions, no longer needed)
    uint32_t* d_rec = d_posi;
    hipLaunchKernelGGL(k_rec_list, dim3(grid_for(nnodes)), dim3(GB), 0, st, nnodes, d_isrec, d_qidx, d_rn, d_rec, d_hdr);
    if (nq)
        hipLaunchKernelGGL(k_records, dim3(grid_for(nq)), dim3(GB), 0, st, nq, d_rec, d_rn, d_qidx, d_qn, d_cn, d_hdr);
    GCHK(hipGetLastError());
    if (nsph) GCHK(hipMemcpyAsync(d_s, srec.data(), sizeof(SphereRec) * nsph, hipMemcpyHostToDevice, st));
    GCHK(hipMemcpyAsync(&hdr, d_hdr, sizeof(hdr), hipMemcpyDeviceToHost, st));
    GCHK(hipStreamSynchronize(st));
    const RNode root = hdr.root;
    const uint32_t bad = hdr.bad_cq;
    SceneView& v = S->view;
    v.rnodes = d_rn;
    v.qnodes = d_qn;
    v.prims = d_pr;
    v.spheres = nsph ? d_s : nullptr;
    const bool cq = nq > 0 && !bad;
    v.cnodes = cq ? d_cn : nullptr;
    v.prims64 = cq ? d_pr64 : nullptr;
    v.ocnodes = v.cnodes;
    v.order = d_order;
    v.n_rnodes = nnodes;
    v.n_qnodes = nq;
    v.n_prims = n;
    v.n_spheres = nsph;
    v.qroot = n > 1 ? 0 : ~(int32_t)0;
    v.ocroot = v.qroot;
    v.depth = maxd;
    v.qdepth = n > 1 ? maxd / 2 + 1 : 0;
    v.odepth = v.qdepth;
    for (int a = 0; a < 3; ++a) { v.root_lo[a] = root.lo[a]; v.root_hi[a] = root.hi[a]; }
    S->bytes = (uint64_t)nnodes * sizeof(RNode) + (uint64_t)nq * (sizeof(QNode) + sizeof(CNode)) +
               (uint64_t)n * (sizeof(PrimRec) + sizeof(PrimRec64) + 4) + (uint64_t)nsph * sizeof(SphereRec);
    *build_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return PBRTX_OK;
}

}  // namespace px

extern "C" int pbrtx_scene_build_gpu(const float* verts, uint32_t nverts, const uint32_t* idx, uint32_t nfaces,
                                     const pbrtx_sphere* spheres, uint32_t nspheres, pbrtx_scene** out,
                                     double* build_ms) {
    using namespace px;
    if (!out) return fail(PBRTX_ERR_ARG, "out is null");
    *out = nullptr;
    static_assert(sizeof(pbrtx_sphere) == sizeof(SphereIn), "sphere layout");
    pbrtx_scene* s = new (std::nothrow) pbrtx_scene();
    if (!s) return fail(PBRTX_ERR_OOM, "host allocation");
    double ms = 0.0;
    int rc = gpu_build_scene(verts, nverts, idx, nfaces, reinterpret_cast<const SphereIn*>(spheres), nspheres, &s->s,
                             &ms);
    if (rc) {
        scene_free(&s->s);
        delete s;
        return rc;
    }
    if (build_ms) *build_ms = ms;
    *out = s;
    return PBRTX_OK;
}
