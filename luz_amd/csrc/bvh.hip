// bvh.hip — BLAS and TLAS builds on gfx950.
//
// Replaces the driver builds behind vkw::CmdBuildBLAS / vkw::CmdBuildTLAS
// (VulkanWrapper.cpp:1089-1104, 1106-1139) with a deterministic LBVH
// (Karras 2012, "Maximizing Parallelism in the Construction of BVHs,
// Octrees, and k-d Trees"):
//   1. padded triangle boxes + FP64 centroid bounds (block reductions);
//   2. 30-bit Morton codes in the FP64 frame;
//   3. stable LSD radix sort, 4 passes of 8 bits: per-tile histograms, one
//      scan, and a scatter that ranks keys inside a tile with wave ballots
//      (8 ballots give each lane the set of lanes holding the same digit);
//   4. Karras hierarchy, one thread per internal node;
//   5. triangle gather into slot order (36-byte records);
//   6. bottom-up refit, one thread per leaf, second arrival continues.
// The TLAS build runs in one workgroup (<= 8192 instances): world boxes,
// FP64 frame, Morton codes, bitonic sort of (code, index) in LDS, Karras,
// refit.  Both produce byte-identical nodes to a sequential CPU build.
#include "internal.hpp"
#include "scan.hpp"

namespace luz {
namespace {

constexpr int kBlock = 256;
constexpr int kSortItems = 16;
constexpr int kSortTile = kBlock * kSortItems;

__device__ inline uint32_t expand10(uint32_t v) {
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}

// Morton code of the FP32 box centroid 0.5 (lo + hi) in the frame {origin[3],
// scale[3]}: the FP64 centroid-bounds reduction rounded to FP32 (morton_frame32).
// Quantisation is FP32; only the reduction that sets the frame runs in FP64.
__device__ inline uint32_t morton_code(const float* frame, const float* box) {
    uint32_t q[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float c = 0.5f * (box[k] + box[3 + k]);
        float t = floorf((c - frame[k]) * frame[3 + k]);
        if (!(t >= 0.0f)) t = 0.0f;
        if (t > 1023.0f) t = 1023.0f;
        q[k] = (uint32_t)t;
    }
    return (expand10(q[0]) << 2) | (expand10(q[1]) << 1) | expand10(q[2]);
}

// The FP32 quantisation frame from the FP64 centroid bounds mn, mx of one
// axis: origin mn and scale 1024 / (mx - mn) (0 for a flat axis), each
// rounded once to FP32.
__device__ inline void morton_frame32(double mn, double mx, float& origin, float& scale) {
    const double e = mx - mn;
    origin = (float)mn;
    scale = e > 0.0 ? (float)(1024.0 / e) : 0.0f;
}

// Padded triangle box (max |coord| * 2^-16 on every side).
__device__ inline void tri_box(V3 a, V3 b, V3 c, float* box) {
    float lo0 = fmin_(fmin_(a.x, b.x), c.x), hi0 = fmax_(fmax_(a.x, b.x), c.x);
    float lo1 = fmin_(fmin_(a.y, b.y), c.y), hi1 = fmax_(fmax_(a.y, b.y), c.y);
    float lo2 = fmin_(fmin_(a.z, b.z), c.z), hi2 = fmax_(fmax_(a.z, b.z), c.z);
    float m = 0.0f;
    m = fmax_(m, fabsf(lo0)); m = fmax_(m, fabsf(hi0));
    m = fmax_(m, fabsf(lo1)); m = fmax_(m, fabsf(hi1));
    m = fmax_(m, fabsf(lo2)); m = fmax_(m, fabsf(hi2));
    float pad = m * 0x1p-16f;
    box[0] = lo0 - pad; box[1] = lo1 - pad; box[2] = lo2 - pad;
    box[3] = hi0 + pad; box[4] = hi1 + pad; box[5] = hi2 + pad;
}

__device__ inline V3 load_pos(const uint8_t* base, uint32_t stride, uint32_t i) {
    const float* p = (const float*)(base + (size_t)i * stride);
    return v3(p[0], p[1], p[2]);
}

template <typename T, typename Op>
__device__ inline T block_reduce(T v, T* sh, Op op) {
    const int tid = threadIdx.x;
    sh[tid] = v;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if (tid < s) sh[tid] = op(sh[tid], sh[tid + s]);
        __syncthreads();
    }
    T r = sh[0];
    __syncthreads();
    return r;
}

struct DMin { __device__ double operator()(double a, double b) const { return b < a ? b : a; } };
struct DMax { __device__ double operator()(double a, double b) const { return b > a ? b : a; } };

// Index of vertex k of triangle t, clamped into range; out-of-range
// indices set the error flag (the build then fails) instead of reading
// outside the vertex buffer.
__device__ inline uint32_t vidx(const uint32_t* idx, uint32_t i, uint32_t nv, uint32_t* error) {
    uint32_t v = idx[i];
    if (v >= nv) { atomicOr(error, 2u); v = 0; }
    return v;
}

__global__ __launch_bounds__(kBlock) void k_tri_boxes(const uint8_t* verts, uint32_t stride,
                                                      uint32_t nv, const uint32_t* idx, uint32_t n,
                                                      float* boxes, double* partial,
                                                      uint32_t* error) {
    __shared__ double sh[kBlock];
    uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    double c[3] = {INFINITY, INFINITY, INFINITY}, C[3] = {-INFINITY, -INFINITY, -INFINITY};
    if (t < n) {
        V3 a = load_pos(verts, stride, vidx(idx, 3 * t, nv, error));
        V3 b = load_pos(verts, stride, vidx(idx, 3 * t + 1, nv, error));
        V3 cc = load_pos(verts, stride, vidx(idx, 3 * t + 2, nv, error));
        float bx[6];
        tri_box(a, b, cc, bx);
#pragma unroll
        for (int k = 0; k < 6; ++k) boxes[(size_t)t * 6 + k] = bx[k];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            double ck = 0.5 * ((double)bx[k] + (double)bx[3 + k]);
            c[k] = ck; C[k] = ck;
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        double mn = block_reduce(c[k], sh, DMin());
        double mx = block_reduce(C[k], sh, DMax());
        if (threadIdx.x == 0) { partial[blockIdx.x * 6 + k] = mn; partial[blockIdx.x * 6 + 3 + k] = mx; }
    }
}

// frame = {cmin[3], scale[3]} with scale = 1024/extent (0 for a flat axis).
__global__ __launch_bounds__(kBlock) void k_frame(const double* partial, uint32_t nparts,
                                                  float* frame) {
    __shared__ double sh[kBlock];
    for (int k = 0; k < 3; ++k) {
        double mn = INFINITY, mx = -INFINITY;
        for (uint32_t i = threadIdx.x; i < nparts; i += kBlock) {
            double a = partial[i * 6 + k], b = partial[i * 6 + 3 + k];
            mn = a < mn ? a : mn;
            mx = b > mx ? b : mx;
        }
        mn = block_reduce(mn, sh, DMin());
        mx = block_reduce(mx, sh, DMax());
        if (threadIdx.x == 0) morton_frame32(mn, mx, frame[k], frame[3 + k]);
    }
}

__global__ __launch_bounds__(kBlock) void k_morton(const float* boxes, uint32_t n,
                                                   const float* frame, uint32_t* keys,
                                                   uint32_t* vals) {
    uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= n) return;
    keys[t] = morton_code(frame, boxes + (size_t)t * 6);
    vals[t] = t;
}

// ---------------------------------------------------------------- radix sort
__global__ __launch_bounds__(kBlock) void k_sort_hist(const uint32_t* keys, uint32_t n,
                                                      int shift, uint32_t* hist,
                                                      uint32_t nblocks) {
    __shared__ uint32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    uint32_t base = blockIdx.x * kSortTile;
    for (int r = 0; r < kSortItems; ++r) {
        uint32_t i = base + r * kBlock + threadIdx.x;
        if (i < n) atomicAdd(&h[(keys[i] >> shift) & 0xFFu], 1u);
    }
    __syncthreads();
    hist[threadIdx.x * nblocks + blockIdx.x] = h[threadIdx.x];
}

// Exclusive scan of the digit counts (16-byte aligned).  A run of consecutive
// counts per thread, read as 16-byte vectors: 200k keys (12,800 counts) 5.7 us
// a pass against 24 us with 1024 counts at a time and twenty barriers each.
__global__ __launch_bounds__(1024) void k_sort_scan(uint32_t* data, uint32_t count) { scan_runs_1024(data, count); }

__global__ __launch_bounds__(kBlock) void k_sort_scatter(const uint32_t* keys_in,
                                                         const uint32_t* vals_in, uint32_t n,
                                                         int shift, const uint32_t* offsets,
                                                         uint32_t nblocks, uint32_t* keys_out,
                                                         uint32_t* vals_out) {
    __shared__ uint32_t digit_base[256];
    __shared__ uint32_t wave_cnt[kBlock / 64][256];
    const int tid = threadIdx.x;
    const int wave = tid >> 6;
    const int lane = tid & 63;
    digit_base[tid] = offsets[tid * nblocks + blockIdx.x];
    for (int w = 0; w < kBlock / 64; ++w) wave_cnt[w][tid] = 0;
    __syncthreads();
    const uint32_t base = blockIdx.x * kSortTile;
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int r = 0; r < kSortItems; ++r) {
        uint32_t i = base + r * kBlock + tid;
        bool valid = i < n;
        uint32_t key = valid ? keys_in[i] : 0u;
        uint32_t val = valid ? vals_in[i] : 0u;
        uint32_t d = (key >> shift) & 0xFFu;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            bool bit = (d >> b) & 1u;
            uint64_t m = __ballot(bit);
            peers &= bit ? m : ~m;
        }
        uint32_t rank = (uint32_t)__popcll(peers & lt);
        if (valid && rank == 0) wave_cnt[wave][d] = (uint32_t)__popcll(peers);
        __syncthreads();
        {
            uint32_t run = digit_base[tid];
            for (int w = 0; w < kBlock / 64; ++w) {
                uint32_t c = wave_cnt[w][tid];
                wave_cnt[w][tid] = run;
                run += c;
            }
            digit_base[tid] = run;
        }
        __syncthreads();
        if (valid) {
            uint32_t pos = wave_cnt[wave][d] + rank;
            keys_out[pos] = key;
            vals_out[pos] = val;
        }
        __syncthreads();
        for (int w = 0; w < kBlock / 64; ++w) wave_cnt[w][tid] = 0;
        __syncthreads();
    }
}

// ---------------------------------------------------------------- hierarchy
__device__ inline int delta_k(const uint32_t* k, int n, int i, int j) {
    if (j < 0 || j > n - 1) return -1;
    uint32_t a = k[i], b = k[j];
    if (a == b) return 32 + __clz((int)((uint32_t)i ^ (uint32_t)j));
    return __clz((int)(a ^ b));
}

// Karras split for internal node i; writes children and parents.
__device__ inline void karras_node(const uint32_t* keys, int n, int i, Node* nodes,
                                   uint32_t* leaf_parent, uint32_t* node_end) {
    int d = (delta_k(keys, n, i, i + 1) - delta_k(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    int dmin = delta_k(keys, n, i, i - d);
    int lmax = 2;
    while (delta_k(keys, n, i, i + lmax * d) > dmin) lmax *= 2;
    int l = 0;
    for (int t = lmax / 2; t >= 1; t /= 2)
        if (delta_k(keys, n, i, i + (l + t) * d) > dmin) l += t;
    int j = i + l * d;
    int dnode = delta_k(keys, n, i, j);
    int s = 0;
    int t = l;
    do {
        t = (t + 1) >> 1;
        if (delta_k(keys, n, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    int gamma = i + s * d + (d < 0 ? d : 0);
    int lo = i < j ? i : j, hi = i < j ? j : i;
    if (node_end) node_end[i] = (uint32_t)j;   // node i covers leaf slots lo..hi
    uint32_t left = (lo == gamma) ? (kLeaf | (uint32_t)gamma) : (uint32_t)gamma;
    uint32_t right = (hi == gamma + 1) ? (kLeaf | (uint32_t)(gamma + 1)) : (uint32_t)(gamma + 1);
    Node& nd = nodes[i];
    nd.child[0] = left;
    nd.child[1] = right;
    nd.pad = 0;
    if (i == 0) nd.parent = kNone;
    if (left & kLeaf) leaf_parent[left & ~kLeaf] = (uint32_t)i; else nodes[left].parent = (uint32_t)i;
    if (right & kLeaf) leaf_parent[right & ~kLeaf] = (uint32_t)i; else nodes[right].parent = (uint32_t)i;
}

__global__ __launch_bounds__(kBlock) void k_karras(const uint32_t* keys, uint32_t n, Node* nodes,
                                                   uint32_t* leaf_parent, uint32_t* node_end,
                                                   uint32_t* counters) {
    uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n - 1) return;
    karras_node(keys, (int)n, (int)i, nodes, leaf_parent, node_end);
    counters[i] = 0;
}

__global__ __launch_bounds__(kBlock) void k_gather(const uint8_t* verts, uint32_t stride,
                                                   uint32_t nv, const uint32_t* idx,
                                                   const uint32_t* order, uint32_t n,
                                                   const float* boxes, float* tris, float* nrms,
                                                   uint32_t* prims, uint32_t* slot_idx,
                                                   float* slot_box, uint32_t* error) {
    uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    if (s >= n) return;
    uint32_t p = order[s];
    prims[s] = p;
    bool has_n = stride >= 24;
#pragma unroll
    for (int v = 0; v < 3; ++v) {
        uint32_t vi = vidx(idx, 3 * p + v, nv, error);
        slot_idx[3 * s + v] = vi;
        const float* q = (const float*)(verts + (size_t)vi * stride);
        tris[(size_t)s * 9 + v * 3 + 0] = q[0];
        tris[(size_t)s * 9 + v * 3 + 1] = q[1];
        tris[(size_t)s * 9 + v * 3 + 2] = q[2];
        nrms[(size_t)s * 9 + v * 3 + 0] = has_n ? q[3] : 0.0f;
        nrms[(size_t)s * 9 + v * 3 + 1] = has_n ? q[4] : 0.0f;
        nrms[(size_t)s * 9 + v * 3 + 2] = has_n ? q[5] : 0.0f;
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) slot_box[(size_t)s * 6 + k] = boxes[(size_t)p * 6 + k];
}

__device__ inline void store_child_box(Node* nd, int side, const float* b) {
    nd->lox[side] = b[0]; nd->loy[side] = b[1]; nd->loz[side] = b[2];
    nd->hix[side] = b[3]; nd->hiy[side] = b[4]; nd->hiz[side] = b[5];
}


constexpr int kRefitChunk = 1024;   // leaf slots per workgroup of the chunk pass
constexpr int kRefitFew = 256;      // the same for one BLAS of a few chunks (launch_refit_chunks)
constexpr uint32_t kRefitFewMax = 16384;
constexpr int kSpanThreads = 1024;  // threads per BLAS of the span pass

// Union of a node's two child boxes, child 0 first (the operand order of
// fmin_/fmax_ matters for signed zeros).
__device__ inline void child_union(int side, const float* mine, const float* other, float* out) {
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const float b0 = side == 0 ? mine[k] : other[k], b1 = side == 0 ? other[k] : mine[k];
        out[k] = k < 3 ? fmin_(b0, b1) : fmax_(b0, b1);
    }
}

__device__ inline uint32_t chunk_job_of(const RefitJob* jobs, uint32_t njobs, uint32_t c) {
    uint32_t lo = 0, hi = njobs;
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (jobs[mid].chunk_offset <= c) lo = mid; else hi = mid;
    }
    return lo;
}

// Chunk pass of a refit (or of a build): one workgroup per CHUNK
// consecutive leaf slots of a BLAS.  Every internal node covers a contiguous
// range of slots that starts or ends at the slot of its own number (Karras), so
// a node whose range lies inside the chunk has both children completed by this
// workgroup: the second child to arrive forms the node's box and writes its two
// child boxes.  A node whose parent's range leaves the chunk stores its box in
// the parent and hands the parent to the span pass through the BLAS's span
// list.  Also zeroes the span pass's arrival counters of the chunk's node ids.
// jobs == nullptr: `single`.
//
// Bound by the length of the climb.  The chunk's part of the hierarchy, the
// arrival counters and the child boxes are in LDS, so a step up waits for no
// global load or store; 1024 slots leave the span pass, which climbs in global
// memory, few nodes.  20,480 triangles: chunk pass 18 -> 22 us, span pass 39 ->
// 23 us against 256-slot chunks with the hierarchy read at every step; 200,978
// triangles 96 -> 38 and 251 -> 66 us (512 slots: 16, 26, 56, 109).
constexpr uint32_t kOutside = 0x80000000u;   // the node's range leaves the chunk
template <bool FROM_VERTS, int CHUNK>
__global__ __launch_bounds__(CHUNK) void k_refit_chunks(const RefitJob* jobs, uint32_t njobs,
                                                              RefitJob single, uint32_t* error) {
    __shared__ uint32_t scnt[CHUNK];
    __shared__ uint2 stopo[CHUNK];   // child 0; parent (31 bits, all set at the root) and kOutside
    __shared__ float sbox[CHUNK * 12];
    const RefitJob& J = jobs ? jobs[chunk_job_of(jobs, njobs, blockIdx.x)] : single;
    const uint32_t c0 = (blockIdx.x - J.chunk_offset) * CHUNK;
    const uint32_t c1 = (c0 + CHUNK < J.n ? c0 + CHUNK : J.n) - 1;   // last slot
    const uint32_t s = c0 + threadIdx.x;
    scnt[threadIdx.x] = 0;
    if (s < J.n - 1) {
        J.counters[s] = 0;
        const uint32_t e = J.node_end[s], up = J.nodes[s].parent;
        const uint32_t lo = s < e ? s : e, hi = s < e ? e : s;
        stopo[threadIdx.x] = make_uint2(J.nodes[s].child[0], (up & ~kOutside) | (lo < c0 || hi > c1 ? kOutside : 0u));
    }
    float box[6];
    uint32_t p = 0;
    if (s < J.n) {
        p = J.leaf_parent[s];
        if (FROM_VERTS) {
            // slot_idx was validated by the build
            V3 v[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) v[k] = load_pos(J.verts, J.stride, J.slot_idx[3 * s + k]);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                J.tris[(size_t)s * 9 + k * 3 + 0] = v[k].x;
                J.tris[(size_t)s * 9 + k * 3 + 1] = v[k].y;
                J.tris[(size_t)s * 9 + k * 3 + 2] = v[k].z;
            }
            tri_box(v[0], v[1], v[2], box);
        } else {
#pragma unroll
            for (int k = 0; k < 6; ++k) box[k] = J.leaf_box[(size_t)s * 6 + k];
        }
    }
    __syncthreads();
    if (s >= J.n) return;
    uint32_t c = kLeaf | s;
    for (int level = 0; p != kNone; ++level) {
        if (level > 80) { atomicOr(error, 1u); return; }
        Node* nd = &J.nodes[p];
        const bool mine = p >= c0 && p <= c1;
        const uint2 t = mine ? stopo[p - c0] : make_uint2(0u, kOutside);
        if (t.y & kOutside) {
            store_child_box(nd, (mine ? t.x : nd->child[0]) == c ? 0 : 1, box);
            const uint32_t k = atomicAdd(&J.span[0], 1u);
            J.span[1 + k] = p;
            return;
        }
        const int side = t.x == c ? 0 : 1;
        float* sb = &sbox[(p - c0) * 12];
#pragma unroll
        for (int k = 0; k < 6; ++k) sb[side * 6 + k] = box[k];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        if (atomicAdd(&scnt[p - c0], 1u) == 0) return;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        float b[2][6];
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            const float other = sb[(1 - side) * 6 + k];
            b[0][k] = side == 0 ? box[k] : other;
            b[1][k] = side == 0 ? other : box[k];
        }
        float4* q = reinterpret_cast<float4*>(nd);
#pragma unroll
        for (int a = 0; a < 3; ++a) q[a] = make_float4(b[0][a], b[1][a], b[0][3 + a], b[1][3 + a]);
        child_union(0, b[0], b[1], box);
        c = p;
        p = t.y == ~kOutside ? kNone : t.y;
    }
}

// Span pass: one workgroup per BLAS completes the nodes whose slot range
// crosses a chunk boundary, climbing from the span list (each entry is one
// arrival at a node whose child box is already stored in it).  Every arrival
// at these nodes comes from this workgroup, so arrival counters in global
// memory with workgroup-scope ordering suffice.  Leaves the list empty.
__global__ __launch_bounds__(kSpanThreads) void k_refit_spans(const RefitJob* jobs, RefitJob single,
                                                              uint32_t* error) {
    const RefitJob& J = jobs ? jobs[blockIdx.x] : single;
    const uint32_t count = J.span[0];
    for (uint32_t i = threadIdx.x; i < count; i += kSpanThreads) {
        uint32_t p = J.span[1 + i];
        for (int level = 0;; ++level) {
            if (level > 80) { atomicOr(error, 1u); break; }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            if (__hip_atomic_fetch_add(&J.counters[p], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == 0)
                break;
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
            const Node* nd = &J.nodes[p];
            const float b0[6] = {nd->lox[0], nd->loy[0], nd->loz[0], nd->hix[0], nd->hiy[0], nd->hiz[0]};
            const float b1[6] = {nd->lox[1], nd->loy[1], nd->loz[1], nd->hix[1], nd->hiy[1], nd->hiz[1]};
            float u[6];
            child_union(0, b0, b1, u);
            const uint32_t q = nd->parent;
            if (q == kNone) break;
            Node* nq = &J.nodes[q];
            store_child_box(nq, nq->child[0] == p ? 0 : 1, u);
            p = q;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) J.span[0] = 0;
}

// BLAS of 0 or 1 triangles: a single root with an empty second child.
__global__ void k_small_root(const uint8_t* verts, uint32_t stride, uint32_t nv,
                             const uint32_t* idx, uint32_t n, Node* nodes, float* tris,
                             float* nrms, uint32_t* prims, uint32_t* slot_idx, uint32_t* error) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    Node nd;
    float empty[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    float b[6];
    if (n == 1) {
        V3 v[3];
        for (int k = 0; k < 3; ++k) {
            uint32_t vi = vidx(idx, k, nv, error);
            slot_idx[k] = vi;
            const float* q = (const float*)(verts + (size_t)vi * stride);
            v[k] = v3(q[0], q[1], q[2]);
            tris[k * 3 + 0] = q[0]; tris[k * 3 + 1] = q[1]; tris[k * 3 + 2] = q[2];
            nrms[k * 3 + 0] = stride >= 24 ? q[3] : 0.0f;
            nrms[k * 3 + 1] = stride >= 24 ? q[4] : 0.0f;
            nrms[k * 3 + 2] = stride >= 24 ? q[5] : 0.0f;
        }
        tri_box(v[0], v[1], v[2], b);
        prims[0] = 0;
    } else {
        for (int k = 0; k < 6; ++k) b[k] = empty[k];
    }
    store_child_box(&nd, 0, b);
    store_child_box(&nd, 1, empty);
    nd.child[0] = n == 1 ? kLeaf : kEmpty;
    nd.child[1] = kEmpty;
    nd.parent = kNone;
    nd.pad = 0;
    nodes[0] = nd;
}

// ---------------------------------------------------------------- 8-wide form
// Collapse of the binary LBVH into 8-wide nodes, numbered breadth first.  The
// eight slots of a wide node depend on its binary root alone, so the long part
// needs no order: k_wide_slots lists them for every binary node at once.  What
// goes level by level is only the numbering (k_wide_number, one workgroup per
// BLAS, or k_wide_level_* with the whole chip for large ones), and k_wide_emit
// then writes all wide nodes together.  One launch of each serves up to
// kWideJobs BLASes and the host waits for none of it.  (With the slots found
// level by level, seven launches and copies and a wait for the host per level,
// five 20,480-triangle meshes took 3.3 ms, now 93 us.)
struct WideJob {
    const Node* bn;
    const uint32_t* leaf_parent;
    const float* tris;
    const uint32_t* prims;
    uint4* slots;          // two per binary node: its 8 slots, left to right (kEmpty: none)
    uint32_t* root;        // per wide node: its binary root
    uint32_t* child_base;  // first child and first triangle of a wide node
    uint32_t* tri_base;
    Node8* out;
    float* tris8;
    uint32_t* prims8;
    uint32_t* count;       // wide nodes
    uint32_t n;            // binary nodes
    uint32_t block, blocks;   // this job's workgroups in a launch over all jobs' nodes
};
constexpr uint32_t kWideJobs = 8;
struct WideJobs {
    uint32_t n, pad;
    WideJob j[kWideJobs];
};

__device__ inline const WideJob& wide_job_of(const WideJobs& J, uint32_t block) {
    uint32_t k = 0;
    while (k + 1 < J.n && J.j[k + 1].block <= block) ++k;
    return J.j[k];
}

__device__ inline float surface_area(const float* lo, const float* hi) {
    float dx = hi[0] - lo[0], dy = hi[1] - lo[1], dz = hi[2] - lo[2];
    return dx * dy + dy * dz + dz * dx;
}

__device__ inline float child_area(const Node& n, int c) {
    const float lo[3] = {n.lox[c], n.loy[c], n.loz[c]}, hi[3] = {n.hix[c], n.hiy[c], n.hiz[c]};
    return surface_area(lo, hi);
}

// The slots of the wide node rooted at each binary node: its two children, then
// repeatedly the internal slot of largest surface area, first on ties, replaced
// in place by its two children.  Bound by the chain of up to six node reads;
// the slots stay in registers (every index is a constant after unrolling).
__global__ __launch_bounds__(kBlock) void k_wide_slots(WideJobs jobs) {
    const WideJob& J = wide_job_of(jobs, blockIdx.x);
    const uint32_t i = (blockIdx.x - J.block) * kBlock + threadIdx.x;
    if (i >= J.n) return;
    uint32_t c[8];
    float sa[8];
    int n = 0;
    {
        const Node nd = J.bn[i];
#pragma unroll
        for (int k = 0; k < 8; ++k) { c[k] = kEmpty; sa[k] = 0.0f; }
        c[0] = nd.child[0];
        sa[0] = child_area(nd, 0);
        n = c[0] != kEmpty ? 1 : 0;
        if (nd.child[1] != kEmpty) {
            c[1] = nd.child[1];
            sa[1] = child_area(nd, 1);
            n = 2;
        }
    }
    while (n < 8) {
        int best = -1;
        float best_sa = 0.0f;
        uint32_t bc = 0;
#pragma unroll
        for (int k = 0; k < 8; ++k)   // kEmpty has the leaf bit
            if (!(c[k] & kLeaf) && (best < 0 || sa[k] > best_sa)) { best = k; best_sa = sa[k]; bc = c[k]; }
        if (best < 0) break;
        const Node nd = J.bn[bc];
        const float a0 = child_area(nd, 0), a1 = child_area(nd, 1);
#pragma unroll
        for (int k = 7; k > 0; --k) {
            if (k > best + 1) { c[k] = c[k - 1]; sa[k] = sa[k - 1]; }
            else if (k == best + 1) { c[k] = nd.child[1]; sa[k] = a1; }
            else if (k == best) { c[k] = nd.child[0]; sa[k] = a0; }
        }
        if (best == 0) { c[0] = nd.child[0]; sa[0] = a0; }
        ++n;
    }
    J.slots[2 * (size_t)i] = make_uint4(c[0], c[1], c[2], c[3]);
    J.slots[2 * (size_t)i + 1] = make_uint4(c[4], c[5], c[6], c[7]);
}

__device__ inline void slot_array(uint4 a, uint4 b, uint32_t (&c)[8]) {
    c[0] = a.x; c[1] = a.y; c[2] = a.z; c[3] = a.w;
    c[4] = b.x; c[5] = b.y; c[6] = b.z; c[7] = b.w;
}

// Internal (low half) and leaf (high half) slots.
__device__ inline uint32_t slot_counts(const uint32_t (&c)[8]) {
    uint32_t k = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) k += c[i] == kEmpty ? 0u : ((c[i] & kLeaf) ? 0x10000u : 1u);
    return k;
}

// Exclusive prefix of v among the workgroup's threads (thread order) and its
// total; the halves of v are summed apart (8 x 1024 fits 16 bits).  sums: one
// word per wave.
__device__ inline uint32_t block_prefix_sum(uint32_t v, uint32_t* sums, uint32_t& total) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t incl = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(incl, off);
        if (lane >= (uint32_t)off) incl += y;
    }
    if (lane == 63) sums[wave] = incl;
    __syncthreads();
    uint32_t before = 0;
    total = 0;
    for (uint32_t w = 0; w < blockDim.x / 64; ++w) {
        const uint32_t t = sums[w];
        if (w < wave) before += t;
        total += t;
    }
    __syncthreads();
    return before + incl - v;
}

// Numbers wide node w (of binary root whose slots are c) given the first child
// and triangle its level has left for it, and lists its children's roots.
__device__ inline void wide_place(const WideJob& J, uint32_t w, const uint32_t (&c)[8], uint32_t child, uint32_t tri) {
    J.child_base[w] = child;
    J.tri_base[w] = tri;
#pragma unroll
    for (int k = 0; k < 8; ++k)
        if (!(c[k] & kLeaf)) J.root[child++] = c[k];
}

// Breadth-first numbering of one BLAS by one workgroup: per level, running
// sums of the nodes' child and triangle counts.  About 2.6 us per 1024 wide
// nodes.  Stops before a level of more than `stop` nodes, left in *level.
__global__ __launch_bounds__(1024) void k_wide_number(WideJobs jobs, uint32_t stop, uint3* level) {
    __shared__ uint32_t sums[1024 / 64];
    const WideJob& J = jobs.j[blockIdx.x];
    if (threadIdx.x == 0) J.root[0] = 0;
    uint32_t start = 0, count = 1, tri = 0;
    while (count > 0 && count <= stop) {
        __syncthreads();   // the level's roots are written
        const uint32_t next = start + count;
        uint32_t children = 0, leaves = 0;
        for (uint32_t base = 0; base < count; base += 1024) {
            const uint32_t i = base + threadIdx.x, w = start + i;
            uint32_t c[8] = {kEmpty, kEmpty, kEmpty, kEmpty, kEmpty, kEmpty, kEmpty, kEmpty};
            if (i < count) {
                const uint32_t r = J.root[w];
                slot_array(J.slots[2 * (size_t)r], J.slots[2 * (size_t)r + 1], c);
            }
            uint32_t total;
            const uint32_t pre = block_prefix_sum(slot_counts(c), sums, total);
            if (i < count) wide_place(J, w, c, next + children + (pre & 0xFFFFu), tri + leaves + (pre >> 16));
            children += total & 0xFFFFu;
            leaves += total >> 16;
        }
        tri += leaves;
        start = next;
        count = children;
    }
    if (threadIdx.x == 0) {
        *J.count = start;
        if (level) *level = make_uint3(start, count, tri);
    }
}

// The wide levels of a large BLAS, one per pair of launches: workgroup b takes
// the b-th run of the level's nodes, k_wide_level_count sums the runs and
// k_wide_level_write numbers them.  levels[l] = (first wide node, nodes, first
// triangle) of level l.
constexpr uint32_t kWideLevelBlocks = 512;
__device__ inline uint32_t level_run(uint32_t count) {
    return (count + kWideLevelBlocks * kBlock - 1) / (kWideLevelBlocks * kBlock) * kBlock;
}

__global__ __launch_bounds__(kBlock) void k_wide_level_count(WideJob J, const uint3* level, uint2* run_sums) {
    __shared__ uint32_t sums[kBlock / 64];
    const uint3 L = *level;
    const uint32_t per = level_run(L.y), begin = blockIdx.x * per;
    const uint32_t end = begin + per < L.y ? begin + per : L.y;
    uint2 s = make_uint2(0u, 0u);
    for (uint32_t base = begin; base < end; base += kBlock) {
        const uint32_t i = base + threadIdx.x;
        uint32_t v = 0, total;
        if (i < end) {
            uint32_t c[8];
            const uint32_t r = J.root[L.x + i];
            slot_array(J.slots[2 * (size_t)r], J.slots[2 * (size_t)r + 1], c);
            v = slot_counts(c);
        }
        block_prefix_sum(v, sums, total);
        s.x += total & 0xFFFFu;
        s.y += total >> 16;
    }
    if (threadIdx.x == 0) run_sums[blockIdx.x] = s;
}

__global__ __launch_bounds__(kBlock) void k_wide_level_write(WideJob J, uint3* level, const uint2* run_sums) {
    __shared__ uint32_t sums[kBlock / 64];
    __shared__ uint32_t s_red[4];   // children, leaves before this run; in the level
    const uint3 L = *level;
    if (L.y == 0) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            level[1] = make_uint3(L.x, 0u, L.z);
            *J.count = L.x;
        }
        return;
    }
    if (threadIdx.x < 4) s_red[threadIdx.x] = 0;
    __syncthreads();
    uint32_t a = 0, b = 0, ta = 0, tb = 0;
    for (uint32_t k = threadIdx.x; k < kWideLevelBlocks; k += kBlock) {
        const uint2 v = run_sums[k];
        ta += v.x;
        tb += v.y;
        if (k < blockIdx.x) { a += v.x; b += v.y; }
    }
    atomicAdd(&s_red[0], a);
    atomicAdd(&s_red[1], b);
    atomicAdd(&s_red[2], ta);
    atomicAdd(&s_red[3], tb);
    __syncthreads();
    const uint32_t next = L.x + L.y;
    uint32_t child = next + s_red[0], tri = L.z + s_red[1];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        level[1] = make_uint3(next, s_red[2], L.z + s_red[3]);
        *J.count = next;
    }
    const uint32_t per = level_run(L.y), begin = blockIdx.x * per;
    const uint32_t end = begin + per < L.y ? begin + per : L.y;
    for (uint32_t base = begin; base < end; base += kBlock) {
        const uint32_t i = base + threadIdx.x;
        uint32_t c[8] = {kEmpty, kEmpty, kEmpty, kEmpty, kEmpty, kEmpty, kEmpty, kEmpty}, total;
        if (i < end) {
            const uint32_t r = J.root[L.x + i];
            slot_array(J.slots[2 * (size_t)r], J.slots[2 * (size_t)r + 1], c);
        }
        const uint32_t pre = block_prefix_sum(slot_counts(c), sums, total);
        if (i < end) wide_place(J, L.x + i, c, child + (pre & 0xFFFFu), tri + (pre >> 16));
        child += total & 0xFFFFu;
        tri += total >> 16;
    }
}

__device__ inline void quant_frame(float lo, float hi, float& origin, int& e) {
    float t = (hi - lo) / 255.0f;
    int e0 = -126, em = -126;
    if (t > 0.0f) frexpf(t, &e0);
    float mag = fabsf(lo) > fabsf(hi) ? fabsf(lo) : fabsf(hi);
    if (mag > 0.0f) frexpf(mag, &em);
    e = e0 > em - 23 ? e0 : em - 23;
    if (e < -126) e = -126;
    for (;;) {
        float sc = ldexpf(1.0f, e);
        origin = floorf(lo / sc) * sc;
        if (origin > lo) origin = origin - sc;
        if (origin + 255.0f * sc >= hi || e >= 127) break;   // (127: a box that is not finite)
        ++e;
    }
}

// Quantised bounds: (v - origin) / 2^e by the exact reciprocal of the scale.
__device__ inline uint32_t quant_lo(float v, float origin, float sc, float inv) {
    float q = floorf((v - origin) * inv);
    q = q < 0.0f ? 0.0f : (q > 255.0f ? 255.0f : q);
    while (q > 0.0f && origin + q * sc > v) q = q - 1.0f;
    return (uint32_t)(uint8_t)q;
}

__device__ inline uint32_t quant_hi(float v, float origin, float sc, float inv) {
    float q = ceilf((v - origin) * inv);
    q = q < 0.0f ? 0.0f : (q > 255.0f ? 255.0f : q);
    while (q < 255.0f && origin + q * sc < v) q = q + 1.0f;
    return (uint32_t)(uint8_t)q;
}

// The earlier of a and b unless b is less or equal: the minimum as a left-to-right
// fold of fmin_ takes it (the last of equal zeros), and likewise the maximum.
template <bool MAX>
__device__ inline float fold8(float v, uint32_t k) {
#pragma unroll
    for (uint32_t off = 1; off < 8; off <<= 1) {
        const float o = __shfl_xor(v, (int)off);
        const float a = (k & off) ? o : v, b = (k & off) ? v : o;
        v = MAX ? fmax_(a, b) : fmin_(a, b);
    }
    return v;
}

// Writes the wide nodes: child boxes (kept by the slots' binary parents)
// quantised in the node's frame, and the leaves' triangles in wide order.
// Eight threads per node, one per slot: the quantisation is most of the work
// (five 20,480-triangle meshes 22 us, 49 with one thread per node).
__global__ __launch_bounds__(kBlock) void k_wide_emit(WideJobs jobs) {
    const WideJob& J = wide_job_of(jobs, blockIdx.x);
    const uint32_t t = (blockIdx.x - J.block) * kBlock + threadIdx.x, k = t & 7u;
    const uint32_t count = *J.count;
    for (uint32_t w = t >> 3; w < count; w += J.blocks * (kBlock / 8)) {
        const uint32_t r = J.root[w];
        const uint32_t c = reinterpret_cast<const uint32_t*>(J.slots)[(size_t)r * 8 + k];
        const bool used = c != kEmpty, leaf = used && (c & kLeaf);
        const uint32_t at = !used || J.n == 1   // (a lone triangle's leaf_parent is not written)
                                ? r
                                : (leaf ? J.leaf_parent[c & ~kLeaf] : J.bn[c].parent);
        const Node& p = J.bn[at];
        const bool second = p.child[0] != c;
        const float lo[3] = {second ? p.lox[1] : p.lox[0], second ? p.loy[1] : p.loy[0], second ? p.loz[1] : p.loz[0]};
        const float hi[3] = {second ? p.hix[1] : p.hix[0], second ? p.hiy[1] : p.hiy[0], second ? p.hiz[1] : p.hiz[0]};
        // this node's lanes, and this slot's rank among the slots of its sort
        const uint32_t group = (threadIdx.x & 63u) & ~7u, below = (1u << k) - 1u;
        const uint32_t leaves = (uint32_t)(__ballot(leaf) >> group) & 0xFFu;
        const uint32_t inner = (uint32_t)(__ballot(used && !leaf) >> group) & 0xFFu;
        const uint32_t tri_base = J.tri_base[w];
        uint8_t* out = reinterpret_cast<uint8_t*>(J.out + w);
        uint32_t meta = 0;
        if (leaf) {
            meta = (uint32_t)__popc(leaves & below);
            const uint32_t slot = c & ~kLeaf, dst = tri_base + meta;
            for (int q = 0; q < 9; ++q) J.tris8[(size_t)dst * 9 + q] = J.tris[(size_t)slot * 9 + q];
            J.prims8[dst] = J.prims[slot];
        } else if (used) {
            meta = 0x80u | (uint32_t)__popc(inner & below);
        }
        out[24 + k] = (uint8_t)meta;
        const uint32_t n = (uint32_t)__popc(leaves | inner);
        float origin[3];
        uint32_t es = n << 24;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const float l = fold8<false>(used ? lo[a] : INFINITY, k), h = fold8<true>(used ? hi[a] : -INFINITY, k);
            int e = 0;
            origin[a] = 0.0f;
            if (n > 0) quant_frame(l, h, origin[a], e);
            es |= ((uint32_t)e & 0xFFu) << (8 * a);
            const float sc = ldexpf(1.0f, (int)(int8_t)e), inv = ldexpf(1.0f, -(int)(int8_t)e);
            out[32 + 8 * a + k] = (uint8_t)(used ? quant_lo(lo[a], origin[a], sc, inv) : 0u);
            out[56 + 8 * a + k] = (uint8_t)(used ? quant_hi(hi[a], origin[a], sc, inv) : 0u);
        }
        if (k == 0) {
            reinterpret_cast<uint4*>(out)[0] = make_uint4(__float_as_uint(origin[0]), __float_as_uint(origin[1]),
                                                          __float_as_uint(origin[2]), es);
            reinterpret_cast<uint2*>(out)[2] = make_uint2(J.child_base[w], tri_base);
        } else if (k == 1) {
            reinterpret_cast<uint4*>(out)[5] = make_uint4(0u, 0u, 0u, 0u);
        }
    }
}

// ---------------------------------------------------------------- TLAS
constexpr int kTlasThreads = 1024;
constexpr int kPlocRadius = 16;                              // clustering search radius (slots)
constexpr int kPlocTile = kTlasThreads + 2 * kPlocRadius;    // staged boxes per neighbour pass

// Threads of a TLAS build launch for m (a power of two >= the instance count):
// four waves up to 64 instances (the neighbour search then gives each cluster
// four threads, one per SIMD, and the barriers stay cheap), else kTlasThreads.
inline uint32_t tlas_threads(uint32_t m) { return m <= 64 ? 256u : (uint32_t)kTlasThreads; }

// Merge cost of two cluster boxes as the tile holds them ((lo.xyz, hi.x) and
// (hi.y, hi.z)): half the surface area of the union, FP32 as written, NaN as
// +inf.
__device__ inline float merge_cost(float4 a, float2 a2, float4 b, float2 b2) {
    const float lx = fmin_(a.x, b.x), ly = fmin_(a.y, b.y), lz = fmin_(a.z, b.z);
    const float hx = fmax_(a.w, b.w), hy = fmax_(a2.x, b2.x), hz = fmax_(a2.y, b2.y);
    const float ex = hx - lx, ey = hy - ly, ez = hz - lz;
    const float c = ex * ey + ey * ez + ez * ex;
    return c == c ? c : INFINITY;
}

// The LDS tile of cluster boxes: slot t holds (lo.x, lo.y, lo.z, hi.x) in
// a[t] and (hi.y, hi.z) in b[t], 24 bytes read by two loads.
struct BoxTile {
    float4* a;
    float2* b;
};
__device__ inline void tile_put(BoxTile T, int t, const float* box) {
    T.a[t] = make_float4(box[0], box[1], box[2], box[3]);
    T.b[t] = make_float2(box[4], box[5]);
}
__device__ inline void tile_get(BoxTile T, int t, float* box) {
    const float4 a = T.a[t];
    const float2 b = T.b[t];
    box[0] = a.x; box[1] = a.y; box[2] = a.z;
    box[3] = a.w; box[4] = b.x; box[5] = b.y;
}

// Part q (< 4) of the neighbour search of cluster i among clusters
// i - kPlocRadius .. i + kPlocRadius (within 0 .. count - 1), from a tile that
// holds cluster c at slot c - base + kPlocRadius: candidates 8q .. 8q + 7 of
// the 32 in index order, their boxes read from LDS together (slots outside
// 0 .. count - 1 are read, as the tile spans them, and skipped).  Keeps in
// (best, bj) the least merge cost, the smaller index on equal cost.
__device__ inline void ploc_part(BoxTile tile, uint32_t i, uint32_t base, uint32_t count, int q, float& best,
                                 uint32_t& bj) {
    const int ti = (int)(i - base) + kPlocRadius;
    const float4 a = tile.a[ti];
    const float2 a2 = tile.b[ti];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int k = 8 * q + u, d = k < kPlocRadius ? k - kPlocRadius : k - kPlocRadius + 1;
        const int j = (int)i + d;
        const float c = merge_cost(a, a2, tile.a[ti + d], tile.b[ti + d]);
        if (j >= 0 && j < (int)count && (bj == kNone || c < best)) { best = c; bj = (uint32_t)j; }
    }
}

// Nearest neighbour of cluster i: least merge cost, the smaller index on
// equal cost.
__device__ inline uint32_t ploc_nearest(BoxTile tile, uint32_t i, uint32_t base, uint32_t count) {
    float best = INFINITY;
    uint32_t bj = kNone;
    for (int q = 0; q < 4; ++q) ploc_part(tile, i, base, count, q, best, bj);
    return bj;
}

// The same search by four consecutive threads (a quad), thread q taking part
// q; the quad's parts combine as (cost, index) pairs, least first, which is
// the order of the one-thread search.  All threads of the wave call it; the
// result is valid in every thread of quad i (i < count).
__device__ inline uint32_t ploc_nearest_quad(BoxTile tile, uint32_t i, uint32_t count) {
    float best = INFINITY;
    uint32_t bj = kNone;
    if (i < count) ploc_part(tile, i, 0, count, (int)(threadIdx.x & 3u), best, bj);
    for (int o = 1; o <= 2; o <<= 1) {
        const float ob = __shfl_xor(best, o);
        const uint32_t oj = __shfl_xor(bj, o);
        if (ob < best || (ob == best && oj < bj)) { best = ob; bj = oj; }
    }
    return bj;
}

// Workgroup barrier ordering LDS accesses only: global stores still in
// flight are not waited for.
__device__ inline void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Exclusive ranks of this thread's head and keep flags among the workgroup's
// threads (thread order), and their totals.  All threads must call it.
// LDS_ONLY: its barrier orders LDS accesses only.
template <bool LDS_ONLY = false>
__device__ inline void block_ranks(bool head, bool keep, uint32_t (*s_wave)[kTlasThreads / 64],
                                   uint32_t& hr, uint32_t& kr, uint32_t& th, uint32_t& tk) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint64_t below = lane ? (~0ull >> (64 - lane)) : 0ull;
    const uint64_t bh = __ballot(head), bk = __ballot(keep);
    if (lane == 0) {
        s_wave[0][wave] = (uint32_t)__popcll(bh);
        s_wave[1][wave] = (uint32_t)__popcll(bk);
    }
    if (LDS_ONLY) lds_barrier();
    else __syncthreads();
    uint32_t oh = 0, ok = 0;
    th = 0;
    tk = 0;
    for (uint32_t w = 0; w < blockDim.x / 64; ++w) {
        const uint32_t ch = s_wave[0][w], ck = s_wave[1][w];
        if (w < wave) { oh += ch; ok += ck; }
        th += ch;
        tk += ck;
    }
    hr = oh + (uint32_t)__popcll(bh & below);
    kr = ok + (uint32_t)__popcll(bk & below);
}

// Node idx joining clusters a (child 0) and b (child 1); the children that are
// nodes get idx as their parent.
__device__ inline void ploc_node(Node* nodes, uint32_t idx, const float* a, const float* b, uint32_t ra,
                                 uint32_t rb) {
    Node nd;
    store_child_box(&nd, 0, a);
    store_child_box(&nd, 1, b);
    nd.child[0] = ra;
    nd.child[1] = rb;
    nd.parent = kNone;
    nd.pad = 0;
    nodes[idx] = nd;
    if (!(ra & kLeaf)) nodes[ra].parent = idx;
    if (!(rb & kLeaf)) nodes[rb].parent = idx;
}

// The same node written without its parent field, which the merge that takes
// the node in sets (kNone for the root, node 0): every byte of a node is then
// stored once, so rounds that create and link nodes need not wait for each
// other's stores.
__device__ inline void ploc_node_unlinked(Node* nodes, uint32_t idx, const float* a, const float* b,
                                          uint32_t ra, uint32_t rb) {
    Node* nd = nodes + idx;
    float4* q = reinterpret_cast<float4*>(nd);
    q[0] = make_float4(a[0], b[0], a[3], b[3]);   // lox[2], hix[2]
    q[1] = make_float4(a[1], b[1], a[4], b[4]);   // loy[2], hiy[2]
    q[2] = make_float4(a[2], b[2], a[5], b[5]);   // loz[2], hiz[2]
    *reinterpret_cast<uint2*>(nd->child) = make_uint2(ra, rb);
    nd->pad = 0;
    if (idx == 0) nd->parent = kNone;
    if (!(ra & kLeaf)) nodes[ra].parent = idx;
    if (!(rb & kLeaf)) nodes[rb].parent = idx;
}

__device__ inline void tlas_build_body(const TlasJob& J, uint32_t* error) {
    const InstIn* in = J.in;
    const uint32_t n = J.n, m = J.m;
    float* wbox = J.wbox;
    Node* nodes = J.nodes;
    InstRec* recs = J.recs;
    InstRec* recs_w = J.recs_w;
    InstAux* aux = J.aux;
    float* w2o_out = J.w2o_out;
    uint32_t* order_out = J.order_out;
    // tlas_lds_bytes(m) bytes, m a power of two >= n: the sort keys, then the
    // clustering's box tile, neighbour and reference arrays in the same memory
    // (within 64 KB for 8192 instances).
    extern __shared__ __align__(16) uint64_t skeys[];
    const int tid = threadIdx.x;
    // launched with 64 threads (one wave, cheap barriers) up to 64 instances,
    // else with kTlasThreads
    const uint32_t nt = blockDim.x;

    // 1. world boxes of the BLAS root boxes, scene magnitude
    float mloc = 0.0f;
    for (uint32_t i = tid; i < n; i += nt) {
        const Node& r = in[i].nodes[0];
        float rlo[3] = {fmin_(r.lox[0], r.lox[1]), fmin_(r.loy[0], r.loy[1]), fmin_(r.loz[0], r.loz[1])};
        float rhi[3] = {fmax_(r.hix[0], r.hix[1]), fmax_(r.hiy[0], r.hiy[1]), fmax_(r.hiz[0], r.hiz[1])};
        float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        for (int c = 0; c < 8; ++c) {
            V3 p = v3((c & 1) ? rhi[0] : rlo[0], (c & 2) ? rhi[1] : rlo[1], (c & 4) ? rhi[2] : rlo[2]);
            V3 w = xform_point(in[i].o2w, p);
            lo[0] = fmin_(lo[0], w.x); hi[0] = fmax_(hi[0], w.x);
            lo[1] = fmin_(lo[1], w.y); hi[1] = fmax_(hi[1], w.y);
            lo[2] = fmin_(lo[2], w.z); hi[2] = fmax_(hi[2], w.z);
        }
        for (int k = 0; k < 3; ++k) {
            mloc = fmax_(mloc, fabsf(lo[k]));
            mloc = fmax_(mloc, fabsf(hi[k]));
            wbox[i * 6 + k] = lo[k];
            wbox[i * 6 + 3 + k] = hi[k];
        }
    }
    // scene magnitude: wave maxima, then the 16 wave values (min/max are exact,
    // so the order of the reduction does not change the result)
    __shared__ float s_red[kTlasThreads / 64];
    __shared__ double s_redd[6][kTlasThreads / 64];
    const uint32_t wave = (uint32_t)tid >> 6, lane = (uint32_t)tid & 63u;
    for (int o = 32; o > 0; o >>= 1) mloc = fmax_(mloc, __shfl_xor(mloc, o));
    if (lane == 0) s_red[wave] = mloc;
    __syncthreads();
    float m_all = 0.0f;
    for (uint32_t w = 0; w < nt / 64; ++w) m_all = fmax_(m_all, s_red[w]);
    const float pad = m_all * 0x1p-14f;
    // 2. padded boxes, FP64 centroid frame
    double cmn[3] = {INFINITY, INFINITY, INFINITY}, cmx[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (uint32_t i = tid; i < n; i += nt) {
        for (int k = 0; k < 3; ++k) {
            float lo = wbox[i * 6 + k] - pad, hi = wbox[i * 6 + 3 + k] + pad;
            wbox[i * 6 + k] = lo;
            wbox[i * 6 + 3 + k] = hi;
            double c = 0.5 * ((double)lo + (double)hi);
            cmn[k] = c < cmn[k] ? c : cmn[k];
            cmx[k] = c > cmx[k] ? c : cmx[k];
        }
    }
    for (int k = 0; k < 3; ++k) {
        for (int o = 32; o > 0; o >>= 1) {
            const double a = __shfl_xor(cmn[k], o), b = __shfl_xor(cmx[k], o);
            cmn[k] = a < cmn[k] ? a : cmn[k];
            cmx[k] = b > cmx[k] ? b : cmx[k];
        }
        if (lane == 0) {
            s_redd[k][wave] = cmn[k];
            s_redd[3 + k][wave] = cmx[k];
        }
    }
    __syncthreads();
    float s_frame[6];
    for (int k = 0; k < 3; ++k) {
        double mn = INFINITY, mx = -INFINITY;
        for (uint32_t w = 0; w < nt / 64; ++w) {
            mn = s_redd[k][w] < mn ? s_redd[k][w] : mn;
            mx = s_redd[3 + k][w] > mx ? s_redd[3 + k][w] : mx;
        }
        morton_frame32(mn, mx, s_frame[k], s_frame[3 + k]);
    }
    // 3. Morton codes, bitonic sort of (code << 32 | index)
    auto sort_key = [&](uint32_t i) -> uint64_t {
        if (i >= n) return ~0ull;
        return ((uint64_t)morton_code(s_frame, wbox + i * 6) << 32) | i;
    };
    if (m <= 64) {
        // one wave sorts in registers: lane i holds key i, partners by xor
        if (tid < 64) {
            uint64_t key = sort_key((uint32_t)tid);
            for (uint32_t k = 2; k <= m; k <<= 1) {
                for (uint32_t j = k >> 1; j > 0; j >>= 1) {
                    const uint32_t lo = __shfl_xor((uint32_t)key, (int)j);
                    const uint32_t hi = __shfl_xor((uint32_t)(key >> 32), (int)j);
                    const uint64_t other = ((uint64_t)hi << 32) | lo;
                    const bool lower = ((uint32_t)tid & j) == 0, up = ((uint32_t)tid & k) == 0;
                    const uint64_t mn = other < key ? other : key, mx = other < key ? key : other;
                    key = lower == up ? mn : mx;
                }
            }
            if ((uint32_t)tid < m) skeys[tid] = key;
        }
        __syncthreads();
    } else {
        for (uint32_t i = tid; i < m; i += nt) skeys[i] = sort_key(i);
        __syncthreads();
    }
    for (uint32_t k = 2; m > 64 && k <= m; k <<= 1) {
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            for (uint32_t i = tid; i < m; i += nt) {
                uint32_t ixj = i ^ j;
                if (ixj > i) {
                    uint64_t a = skeys[i], b = skeys[ixj];
                    bool up = (i & k) == 0;
                    if ((a > b) == up) { skeys[i] = b; skeys[ixj] = a; }
                }
            }
            __syncthreads();
        }
    }
    // 4. leaf records in slot order; the clusters start as the leaves
    float* cb = J.cbox[0];
    float* cb2 = J.cbox[1];
    uint32_t* cr = J.cref[0];
    uint32_t* cr2 = J.cref[1];
    for (uint32_t s = tid; s < n; s += nt) {
        uint32_t i = (uint32_t)(skeys[s] & 0xFFFFFFFFu);
        const InstIn& src = in[i];
        InstRec rec;
        for (int k = 0; k < 12; ++k) rec.w2o[k] = src.w2o[k];
        rec.nodes = src.nodes;
        rec.tris = src.tris;
        recs[s] = rec;
        if (recs_w) {
            rec.nodes = reinterpret_cast<const Node*>(src.wnodes);
            rec.tris = src.wtris;
            recs_w[s] = rec;
        }
        InstAux ax;
        for (int k = 0; k < 9; ++k) ax.nmat[k] = src.nmat[k];
        ax.custom_index = src.custom_index;
        ax.input_index = src.input_index;
        ax.pad = 0;
        ax.nrms = src.nrms;
        ax.prims = src.prims;
        aux[s] = ax;
        for (int k = 0; k < 12; ++k) w2o_out[s * 12 + k] = src.w2o[k];
        order_out[s] = src.input_index;
        for (int k = 0; k < 6; ++k) cb[s * 6 + k] = wbox[i * 6 + k];
        for (int k = 0; k < 6; ++k) J.slot_box[s * 6 + k] = wbox[i * 6 + k];
        cr[s] = kLeaf | s;
    }
    __syncthreads();   // the sort keys are dead from here on
    if (n >= 2) {
        // 5. locally-ordered clustering (PLOC, Meister & Bittner 2018): each
        // round every cluster finds the neighbour within kPlocRadius slots of
        // least merge cost, mutual pairs merge into a new node at the lower
        // position, and the survivors are compacted in order.  New nodes are
        // numbered downwards from n - 2 in merge order, so the root is node 0.
        BoxTile tile{reinterpret_cast<float4*>(skeys), nullptr};   // kPlocTile boxes
        tile.b = reinterpret_cast<float2*>(tile.a + kPlocTile);
        uint32_t* snn = reinterpret_cast<uint32_t*>(tile.b + kPlocTile);   // m entries
        uint32_t* sref = snn + m;                                              // kTlasThreads entries
        __shared__ uint32_t s_wave[2][kTlasThreads / 64];
        uint32_t count = n, next = n - 1;
        bool failed = false;
        // rounds over more clusters than threads: cluster arrays in global memory
        while (count > nt && !failed) {
            for (uint32_t base = 0; base < count; base += nt) {
                for (int t = tid; t < (int)nt + 2 * kPlocRadius; t += (int)nt) {
                    const int c = (int)base - kPlocRadius + t;
                    if (c >= 0 && c < (int)count) tile_put(tile, t, cb + (size_t)c * 6);
                }
                __syncthreads();
                const uint32_t i = base + tid;
                if (i < count) snn[i] = ploc_nearest(tile, i, base, count);
                __syncthreads();
            }
            uint32_t heads = 0, kept = 0;
            for (uint32_t base = 0; base < count; base += nt) {
                const uint32_t i = base + tid;
                bool head = false, keep = false;
                uint32_t j = 0;
                if (i < count) {
                    j = snn[i];
                    const bool mutual = snn[j] == i;
                    head = mutual && i < j;
                    keep = !(mutual && i > j);
                }
                uint32_t hr, kr, th, tk;
                block_ranks(head, keep, s_wave, hr, kr, th, tk);
                hr += heads;
                kr += kept;
                if (head) {
                    const uint32_t idx = next - 1 - hr;
                    ploc_node(nodes, idx, cb + (size_t)i * 6, cb + (size_t)j * 6, cr[i], cr[j]);
                    cr2[kr] = idx;
                    for (int k = 0; k < 3; ++k) {
                        cb2[kr * 6 + k] = fmin_(cb[i * 6 + k], cb[j * 6 + k]);
                        cb2[kr * 6 + 3 + k] = fmax_(cb[i * 6 + 3 + k], cb[j * 6 + 3 + k]);
                    }
                } else if (keep) {
                    cr2[kr] = cr[i];
                    for (int k = 0; k < 6; ++k) cb2[kr * 6 + k] = cb[i * 6 + k];
                }
                heads += th;
                kept += tk;
                __syncthreads();
            }
            failed = heads == 0;   // cannot happen: the least-cost pair is mutual
            count = kept;
            next -= heads;
            float* tb = cb; cb = cb2; cb2 = tb;
            uint32_t* tr = cr; cr = cr2; cr2 = tr;
        }
        // rounds over at most one cluster per thread: cluster i lives in thread
        // i's registers and in the LDS tile (box at i + kPlocRadius) and sref;
        // the nodes these rounds create are only stored, so their barriers
        // order LDS accesses alone
        float box[6];
        uint32_t ref = 0;
        if (tid < count) {
            for (int k = 0; k < 6; ++k) box[k] = cb[tid * 6 + k];
            tile_put(tile, tid + kPlocRadius, box);
            ref = cr[tid];
            sref[tid] = ref;
        }
        __syncthreads();
        while (count > 1 && !failed) {
            if (4 * count <= nt) {   // four threads per cluster
                const uint32_t i = (uint32_t)tid >> 2, b = ploc_nearest_quad(tile, i, count);
                if (i < count && (tid & 3) == 0) snn[i] = b;
            } else if (tid < count) {
                snn[tid] = ploc_nearest(tile, tid, 0, count);
            }
            lds_barrier();
            bool head = false, keep = false;
            uint32_t j = 0;
            if (tid < count) {
                j = snn[tid];
                const bool mutual = snn[j] == tid;
                head = mutual && tid < j;
                keep = !(mutual && tid > j);
            }
            uint32_t hr, kr, heads, kept;
            block_ranks<true>(head, keep, s_wave, hr, kr, heads, kept);
            if (head) {
                const uint32_t idx = next - 1 - hr;
                float other[6];
                tile_get(tile, j + kPlocRadius, other);
                ploc_node_unlinked(nodes, idx, box, other, ref, sref[j]);
                for (int k = 0; k < 3; ++k) {
                    box[k] = fmin_(box[k], other[k]);
                    box[3 + k] = fmax_(box[3 + k], other[3 + k]);
                }
                ref = idx;
            }
            lds_barrier();   // every read of this round's tile and sref is done
            if (keep) {
                tile_put(tile, kr + kPlocRadius, box);
                sref[kr] = ref;
            }
            lds_barrier();
            failed = heads == 0;
            count = kept;
            next -= heads;
            if (tid < count) {
                tile_get(tile, tid + kPlocRadius, box);
                ref = sref[tid];
            }
        }
        if (failed && tid == 0) atomicOr(error, 1u);
    } else if (tid == 0) {
        Node nd;
        float empty[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
        if (n == 1) store_child_box(&nd, 0, wbox);
        else store_child_box(&nd, 0, empty);
        store_child_box(&nd, 1, empty);
        nd.child[0] = n == 1 ? kLeaf : kEmpty;
        nd.child[1] = kEmpty;
        nd.parent = kNone;
        nd.pad = 0;
        nodes[0] = nd;
    }
}

__global__ __launch_bounds__(kTlasThreads) void k_tlas_build(TlasJob J, uint32_t* error) {
    tlas_build_body(J, error);
}

// Many TLASes in one launch: workgroup i builds jobs[i].
__global__ __launch_bounds__(kTlasThreads) void k_tlas_build_batched(const TlasJob* jobs,
                                                                     uint32_t* error) {
    tlas_build_body(jobs[blockIdx.x], error);
}

// Batched refit: global triangle t belongs to the job whose tri_offset range holds it.
inline uint32_t cdiv(uint64_t a, uint32_t b) { return (uint32_t)((a + b - 1) / b); }

}  // namespace

// Device flag set by build kernels on bad input or a malformed tree; read by
// luzrt_get_timings / the build call's own check.
uint32_t* build_error_flag(luzrt_ctx* ctx) {
    if (ensure(ctx, ctx->counters, kCounterBytes) != LUZRT_OK) return nullptr;
    return (uint32_t*)ctx->counters.ptr + kCntBuildError;
}

namespace {

// The chunk pass of one BLAS.  Up to 1024 triangles are one chunk with nothing
// left for the span pass.  A few chunks of 1024 slots put their sixteen waves
// each on a few CUs, where they climb in turns, and the span pass has little to
// save: refits (256 / 1024 slots) of 1,800 triangles 23.6 / 30.8 us, 5,000 29.3 /
// 35.9, 9,800 35.4 / 40.9, 20,000 45.0 / 44.2, 80,000 118 / 57; of 800 21.0 / 18.3.
template <bool FROM_VERTS>
void launch_refit_chunks(hipStream_t st, const RefitJob& J, uint32_t* error) {
    if (J.n > (uint32_t)kRefitChunk && J.n <= kRefitFewMax)
        k_refit_chunks<FROM_VERTS, kRefitFew><<<cdiv(J.n, kRefitFew), kRefitFew, 0, st>>>(nullptr, 1, J, error);
    else
        k_refit_chunks<FROM_VERTS, kRefitChunk><<<refit_chunks(J.n), kRefitChunk, 0, st>>>(nullptr, 1, J, error);
}

}  // namespace

luzrt_status blas_build_device(luzrt_ctx* ctx, luzrt_blas* b, const void* vertices,
                               const uint32_t* indices) {
    ctx->release_clean = false;   // BLAS data written on the context's stream
    hipStream_t st = ctx->stream;
    uint32_t* error = build_error_flag(ctx);
    if (!error) return fail(ctx, LUZRT_E_OUT_OF_MEMORY, "no device memory for the error flag");
    const uint32_t n = b->tri_count;
    const uint8_t* verts = (const uint8_t*)vertices;
    if (n <= 1) {
        k_small_root<<<1, 64, 0, st>>>(verts, b->stride, b->vertex_count, indices, n, b->nodes,
                                       b->tris, b->nrms, b->prims, b->slot_idx, error);
        LUZ_HIP(ctx, hipGetLastError());
        return LUZRT_OK;
    }
    const uint32_t nb = cdiv(n, kBlock);
    const uint32_t sb = cdiv(n, kSortTile);
    // 10 sub-allocations, each rounded up to 256 bytes
    size_t bytes = (size_t)n * 24 + (size_t)nb * 48 + 64 + (size_t)n * 16 + (size_t)256 * sb * 4 +
                   (size_t)n * 24 + 10 * 256;
    uint8_t* scratch = nullptr;
    LUZ_HIP(ctx, hipMallocAsync((void**)&scratch, bytes, st));
    uint8_t* p = scratch;
    auto take = [&](size_t sz) { uint8_t* r = p; p += (sz + 255) & ~(size_t)255; return r; };
    float* boxes = (float*)take((size_t)n * 24);
    double* partial = (double*)take((size_t)nb * 48);
    float* frame = (float*)take(64);
    uint32_t* k0 = (uint32_t*)take((size_t)n * 4);
    uint32_t* v0 = (uint32_t*)take((size_t)n * 4);
    uint32_t* k1 = (uint32_t*)take((size_t)n * 4);
    uint32_t* v1 = (uint32_t*)take((size_t)n * 4);
    uint32_t* hist = (uint32_t*)take((size_t)256 * sb * 4);
    float* slot_box = (float*)take((size_t)n * 24);
    (void)bytes;

    k_tri_boxes<<<nb, kBlock, 0, st>>>(verts, b->stride, b->vertex_count, indices, n, boxes, partial,
                                       error);
    k_frame<<<1, kBlock, 0, st>>>(partial, nb, frame);
    k_morton<<<nb, kBlock, 0, st>>>(boxes, n, frame, k0, v0);
    uint32_t *kin = k0, *vin = v0, *kout = k1, *vout = v1;
    for (int pass = 0; pass < 4; ++pass) {
        int shift = pass * 8;
        k_sort_hist<<<sb, kBlock, 0, st>>>(kin, n, shift, hist, sb);
        k_sort_scan<<<1, 1024, 0, st>>>(hist, 256 * sb);
        k_sort_scatter<<<sb, kBlock, 0, st>>>(kin, vin, n, shift, hist, sb, kout, vout);
        std::swap(kin, kout);
        std::swap(vin, vout);
    }
    k_karras<<<cdiv(n - 1, kBlock), kBlock, 0, st>>>(kin, n, b->nodes, b->leaf_parent, b->node_end,
                                                      b->counters);
    k_gather<<<nb, kBlock, 0, st>>>(verts, b->stride, b->vertex_count, indices, vin, n, boxes,
                                    b->tris, b->nrms, b->prims, b->slot_idx, slot_box, error);
    const RefitJob J = refit_job(b, nullptr, slot_box);
    launch_refit_chunks<false>(st, J, error);
    k_refit_spans<<<1, kSpanThreads, 0, st>>>(nullptr, J, error);
    LUZ_HIP(ctx, hipGetLastError());
    LUZ_HIP(ctx, hipFreeAsync(scratch, st));
    return LUZRT_OK;
}

luzrt_status blas_refit_device(luzrt_ctx* ctx, luzrt_blas* b, const void* vertices) {
    ctx->release_clean = false;   // BLAS data written on the context's stream
    hipStream_t st = ctx->stream;
    uint32_t* error = build_error_flag(ctx);
    if (!error) return fail(ctx, LUZRT_E_OUT_OF_MEMORY, "no device memory for the error flag");
    const uint32_t n = b->tri_count;
    if (n <= 1) {
        // rebuild the single root (indices are kept in slot order)
        k_small_root<<<1, 64, 0, st>>>((const uint8_t*)vertices, b->stride, b->vertex_count,
                                       b->slot_idx, n, b->nodes, b->tris, b->nrms, b->prims,
                                       b->slot_idx, error);
        LUZ_HIP(ctx, hipGetLastError());
        return LUZRT_OK;
    }
    const RefitJob J = refit_job(b, vertices, nullptr);
    launch_refit_chunks<true>(st, J, error);
    k_refit_spans<<<1, kSpanThreads, 0, st>>>(nullptr, J, error);
    LUZ_HIP(ctx, hipGetLastError());
    return LUZRT_OK;
}

namespace {

// Bytes of a job's work arrays (slots, roots, child and triangle bases).
size_t wide_work_bytes(uint32_t nodes) { return ((size_t)nodes * 44 + 255) & ~(size_t)255; }

// Above this many binary nodes a BLAS is numbered with the whole chip.
constexpr uint32_t kWideOneGroup = 1u << 17;
// Work arrays up to this size are kept by the context for the next build (an
// animated scene makes one per frame); larger ones are given back.
constexpr size_t kWideKeptBytes = 32u << 20;

luzrt_status wide_number_large(luzrt_ctx* ctx, const WideJob& J, uint8_t* level_mem) {
    hipStream_t st = ctx->stream;
    uint3* level = reinterpret_cast<uint3*>(level_mem);
    uint2* sums = reinterpret_cast<uint2*>(level_mem + 1024);
    // the narrow levels by one workgroup, the wide ones by the whole chip; the
    // host looks whether the tree has ended after as many as most trees have
    WideJobs one{};
    one.n = 1;
    one.j[0] = J;
    k_wide_number<<<1, 1024, 0, st>>>(one, 4096u, level);
    uint32_t done = 0;
    for (uint32_t upto = 4; upto <= 64; upto += 4) {
        for (; done < upto; ++done) {
            k_wide_level_count<<<kWideLevelBlocks, kBlock, 0, st>>>(J, level + done, sums);
            k_wide_level_write<<<kWideLevelBlocks, kBlock, 0, st>>>(J, level + done, sums);
        }
        uint3 last;
        LUZ_HIP(ctx, hipGetLastError());
        LUZ_HIP(ctx, hipMemcpyAsync(&last, level + done, sizeof(last), hipMemcpyDeviceToHost, st));
        LUZ_HIP(ctx, hipStreamSynchronize(st));
        if (last.y == 0) return LUZRT_OK;
    }
    return fail(ctx, LUZRT_E_DEVICE, "8-wide collapse: deeper than 64 levels");
}

// Collapses up to kWideJobs BLASes on the context's stream.
luzrt_status wide_build_some(luzrt_ctx* ctx, luzrt_blas* const* list, uint32_t count) {
    hipStream_t st = ctx->stream;
    constexpr size_t kLevelBytes = 1024 + kWideLevelBlocks * sizeof(uint2);
    size_t bytes = kLevelBytes;
    for (uint32_t k = 0; k < count; ++k) bytes += wide_work_bytes(list[k]->node_count);
    uint8_t* work = nullptr;
    const bool kept = bytes <= kWideKeptBytes;
    if (kept) {
        luzrt_status s = ensure(ctx, ctx->wide_work, bytes);
        if (s != LUZRT_OK) return s;
        work = (uint8_t*)ctx->wide_work.ptr;
    } else {
        LUZ_HIP(ctx, hipMallocAsync((void**)&work, bytes, st));
    }
    uint8_t* p = work + kLevelBytes;
    WideJobs jobs{};
    jobs.n = count;
    uint32_t blocks = 0, small = 0;
    for (uint32_t k = 0; k < count; ++k) {
        luzrt_blas* b = list[k];
        WideJob& J = jobs.j[k];
        J.bn = b->nodes;
        J.leaf_parent = b->leaf_parent;
        J.tris = b->tris;
        J.prims = b->prims;
        J.n = b->node_count;
        J.slots = (uint4*)p;
        J.root = (uint32_t*)(p + (size_t)J.n * 32);
        J.child_base = J.root + J.n;
        J.tri_base = J.child_base + J.n;
        p += wide_work_bytes(J.n);
        J.out = b->wide;
        J.tris8 = b->tris8;
        J.prims8 = b->prims8;
        J.count = b->wide_count_dev;
        J.block = blocks;
        J.blocks = cdiv(J.n, kBlock);
        blocks += J.blocks;
        if (J.n <= kWideOneGroup) ++small;
    }
    k_wide_slots<<<blocks, kBlock, 0, st>>>(jobs);
    luzrt_status s = LUZRT_OK;
    if (small == count) {
        k_wide_number<<<count, 1024, 0, st>>>(jobs, ~0u, nullptr);
    } else {
        WideJobs few{};
        for (uint32_t k = 0; k < count; ++k)
            if (jobs.j[k].n <= kWideOneGroup) few.j[few.n++] = jobs.j[k];
        if (few.n) k_wide_number<<<few.n, 1024, 0, st>>>(few, ~0u, nullptr);
        for (uint32_t k = 0; k < count && s == LUZRT_OK; ++k)
            if (jobs.j[k].n > kWideOneGroup) s = wide_number_large(ctx, jobs.j[k], work);
    }
    if (s == LUZRT_OK) {
        k_wide_emit<<<blocks, kBlock, 0, st>>>(jobs);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) s = hip_fail(ctx, e, "8-wide collapse");
    }
    if (!kept) {
        hipError_t e = hipFreeAsync(work, st);
        if (e != hipSuccess && s == LUZRT_OK) s = hip_fail(ctx, e, "hipFreeAsync");
    }
    if (s != LUZRT_OK) return s;
    for (uint32_t k = 0; k < count; ++k) {
        list[k]->wide_valid = true;
        list[k]->wide_counted = false;
    }
    return LUZRT_OK;
}

}  // namespace

luzrt_status blas_wide_device(luzrt_ctx* ctx, luzrt_blas* const* list, uint32_t count) {
    ctx->release_clean = false;   // BLAS data written on the context's stream
    for (uint32_t k = 0; k < count; ++k) {
        luzrt_blas* b = list[k];
        const size_t n = b->tri_count ? b->tri_count : 1;
        if (b->wide_mem) continue;
        ArrayBlock block;
        const size_t wide = block.add((size_t)b->node_count * sizeof(Node8));   // wide nodes <= binary internal nodes
        const size_t tris8 = block.add(n * 36), prims8 = block.add(n * 4), counted = block.add(4);
        LUZ_HIP(ctx, hipMalloc(&b->wide_mem, block.bytes));
        place(&b->wide, b->wide_mem, wide);
        place(&b->tris8, b->wide_mem, tris8);
        place(&b->prims8, b->wide_mem, prims8);
        place(&b->wide_count_dev, b->wide_mem, counted);
    }
    for (uint32_t k = 0; k < count; k += kWideJobs) {
        luzrt_status s = wide_build_some(ctx, list + k, count - k < kWideJobs ? count - k : kWideJobs);
        if (s != LUZRT_OK) return s;
    }
    return LUZRT_OK;
}

luzrt_status blas_wide_count(luzrt_ctx* ctx, luzrt_blas* b, uint32_t* count) {
    if (!b->wide_counted) {
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        LUZ_HIP(ctx, hipStreamIsCapturing(ctx->stream, &cs));
        if (cs != hipStreamCaptureStatusNone)
            return fail(ctx, LUZRT_E_UNSUPPORTED, "the 8-wide node count cannot be read while the stream is captured");
        LUZ_HIP(ctx, hipMemcpyAsync(&b->wide_count, b->wide_count_dev, 4, hipMemcpyDeviceToHost, ctx->stream));
        LUZ_HIP(ctx, hipStreamSynchronize(ctx->stream));
        b->wide_counted = true;
    }
    *count = b->wide_count;
    return LUZRT_OK;
}

luzrt_status launch_tlas_batched(luzrt_ctx* ctx, const TlasJob* dev_jobs, uint32_t njobs,
                                 uint32_t max_m) {
    uint32_t* error = build_error_flag(ctx);
    if (!error) return fail(ctx, LUZRT_E_OUT_OF_MEMORY, "no device memory for the error flag");
    const size_t lds = tlas_lds_bytes(max_m);
    k_tlas_build_batched<<<njobs, tlas_threads(max_m), lds, ctx->stream>>>(dev_jobs, error);
    LUZ_HIP(ctx, hipGetLastError());
    return LUZRT_OK;
}

uint32_t refit_chunks(uint32_t tris) { return cdiv(tris, kRefitChunk); }

RefitJob refit_job(luzrt_blas* b, const void* vertices, const float* leaf_box) {
    RefitJob J;
    J.nodes = b->nodes;
    J.leaf_parent = b->leaf_parent;
    J.counters = b->counters;
    J.node_end = b->node_end;
    J.span = b->span;
    J.slot_idx = b->slot_idx;
    J.tris = b->tris;
    J.verts = (const uint8_t*)vertices;
    J.leaf_box = leaf_box;
    J.stride = b->stride;
    J.n = b->tri_count;
    J.chunk_offset = 0;
    J.pad = 0;
    return J;
}

luzrt_status launch_refit_batched(luzrt_ctx* ctx, const RefitJob* dev_jobs, uint32_t njobs,
                                  uint32_t total_chunks) {
    uint32_t* error = build_error_flag(ctx);
    if (!error) return fail(ctx, LUZRT_E_OUT_OF_MEMORY, "no device memory for the error flag");
    if (njobs == 0 || total_chunks == 0) return LUZRT_OK;
    RefitJob none{};
    k_refit_chunks<true, kRefitChunk><<<total_chunks, kRefitChunk, 0, ctx->stream>>>(dev_jobs, njobs, none, error);
    k_refit_spans<<<njobs, kSpanThreads, 0, ctx->stream>>>(dev_jobs, none, error);
    LUZ_HIP(ctx, hipGetLastError());
    return LUZRT_OK;
}

// world boxes, two cluster-box planes, two reference planes, slot boxes
size_t tlas_scratch_bytes(uint32_t capacity) {
    return (size_t)capacity * (4 * 6 * sizeof(float) + 2 * sizeof(uint32_t));
}

size_t tlas_lds_bytes(uint32_t m) {
    const size_t sort = (size_t)(m > 1024 ? m : 1024) * sizeof(uint64_t);
    const size_t ploc = (size_t)kPlocTile * (sizeof(float4) + sizeof(float2)) + ((size_t)m + kTlasThreads) * sizeof(uint32_t);
    return sort > ploc ? sort : ploc;
}

TlasJob tlas_job(luzrt_tlas* t, const InstIn* dev_in, uint32_t n) {
    uint32_t m = 1;
    while (m < n) m <<= 1;
    TlasJob J;
    J.in = dev_in;
    J.n = n;
    J.m = m;
    const size_t cap = t->capacity;
    J.wbox = (float*)t->scratch;
    J.cbox[0] = J.wbox + cap * 6;
    J.cbox[1] = J.cbox[0] + cap * 6;
    J.cref[0] = (uint32_t*)(J.cbox[1] + cap * 6);
    J.cref[1] = J.cref[0] + cap;
    J.nodes = t->nodes;
    J.recs = t->recs;
    J.recs_w = t->wide ? t->recs_w : nullptr;
    J.aux = t->aux;
    J.w2o_out = t->w2o;
    J.order_out = t->order;
    J.slot_box = reinterpret_cast<float*>(J.cref[1] + cap);
    return J;
}

const float* tlas_slot_boxes(const luzrt_tlas* t) {
    const size_t cap = t->capacity;
    return reinterpret_cast<const float*>(reinterpret_cast<const uint32_t*>(
                                              reinterpret_cast<const float*>(t->scratch) + cap * 18) +
                                          2 * cap);
}

luzrt_status tlas_build_device(luzrt_ctx* ctx, luzrt_tlas* t, const InstIn* dev_in, uint32_t n,
                               hipStream_t st) {
    uint32_t* error = build_error_flag(ctx);
    if (!error) return fail(ctx, LUZRT_E_OUT_OF_MEMORY, "no device memory for the error flag");
    TlasJob J = tlas_job(t, dev_in, n);
    const size_t lds = tlas_lds_bytes(J.m);
    k_tlas_build<<<1, tlas_threads(J.m), lds, st>>>(J, error);
    LUZ_HIP(ctx, hipGetLastError());
    return LUZRT_OK;
}

}  // namespace luz
