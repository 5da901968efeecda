// traverse.hpp — two-level BVH traversal state machine for gfx950.
//
// One lane owns one ray.  Its stack lives in LDS (kShort entries per lane,
// interleaved so that lane i of a wave touches bank i) and spills its oldest
// entries to a per-lane global array when it overflows, so the depth is
// unbounded by LDS size.  A sentinel entry on the stack marks the return from
// a BLAS to the TLAS (the instance's object-space ray is then dropped).
//
// The step function advances a ray by one node visit (two slab tests, and the
// triangle tests of leaf children) so that a persistent kernel can interleave
// steps with wave-wide refills of finished lanes.
#pragma once
#include "device_math.hpp"

namespace luz {

constexpr int kShort = 16;    // default LDS stack entries per lane (power of two)
constexpr int kSpill = 160;   // global overflow entries per lane (>= TLAS+BLAS depth + 1)

typedef uint32_t __attribute__((address_space(3))) LdsWord;
typedef uint32_t __attribute__((address_space(1))) GlobalWord;

// SHORT: LDS entries per lane (a power of two, chosen by the autotuner);
// DEPTH: the deepest stack a ray may use (its spill column holds DEPTH
// entries).  The two columns carry their address spaces, so a pop reads LDS
// with an LDS load and only an overflowed entry with a global load (a generic
// pointer would turn every pop into a flat load that waits on both memory
// counters).
template <int SHORT, int DEPTH = kSpill>
struct StackT {
    LdsWord* ls;      // this lane's LDS column; entry e at ls[e * lds_stride]
    GlobalWord* gs;   // this lane's spill column; entry e at gs[e * g_stride]
    uint32_t lds_stride;
    uint32_t g_stride;
    int sp, lo;

    __device__ inline void init(uint32_t* lds_column, uint32_t lds_step, uint32_t* spill_column,
                                uint32_t spill_step) {
        ls = (LdsWord*)lds_column;
        gs = (GlobalWord*)spill_column;
        lds_stride = lds_step;
        g_stride = spill_step;
        sp = 0;
        lo = 0;
    }

    // A full stack (DEPTH entries) refuses the push before anything spills, so
    // the spill column is written at entries 0 .. DEPTH - SHORT - 1 only.
    __device__ inline bool push(uint32_t x) {
        if (sp >= DEPTH) return false;
        if (sp - lo == SHORT) {
            gs[(size_t)lo * g_stride] = ls[(lo & (SHORT - 1)) * lds_stride];
            lo++;
        }
        ls[(sp & (SHORT - 1)) * lds_stride] = x;
        sp++;
        return true;
    }
    __device__ inline uint32_t pop() {
        sp--;
        if (sp < lo) {
            lo = sp;
            return gs[(size_t)sp * g_stride];
        }
        return ls[(sp & (SHORT - 1)) * lds_stride];
    }
};
using Stack = StackT<kShort>;

struct Best {
    float t;
    uint32_t inst_slot, tri_slot;
    float T, det, U, V, W;
    bool found;
};

struct RayState {
    V3 wd;         // world direction (the world origin is wbr.o)
    float tmin, tmax;
    BoxRay br;     // the object-space slab-test ray of the instance being walked
    BoxRay wbr;    // the world-space one (TLAS nodes)
    TriRay tr;
    const Node* bnodes;
    const float* btris;
    uint32_t inst_slot;
    uint32_t next;
    uint32_t steps;
    int base;      // TLAS-free rays: the stack below the BLAS being walked
    bool in_blas;
};

// A well-formed two-level tree visits each node at most once per instance
// entry; the cap only guards against a malformed structure looping forever.
constexpr uint32_t kMaxSteps = 1u << 24;

enum StepResult { kStepContinue = 0, kStepHit = 1, kStepDone = 2, kStepOverflow = 3 };

// WIDE: the range of the object-space slab rays is 2^-24 of the ray's (wide_visit).
template <bool WIDE = false, typename STACK>
__device__ inline void ray_begin(RayState& r, STACK& st, V3 o, V3 d, float tmin, float tmax) {
    r.wd = d; r.tmin = tmin; r.tmax = tmax;
    r.wbr = box_setup(o, d, tmin, tmax);
    r.br = r.wbr;
    if (WIDE) {
        r.br.tlo *= 0x1p-24f;
        r.br.thi *= 0x1p-24f;
    }
    r.next = 0;
    r.steps = 0;
    r.in_blas = false;
    st.sp = 0; st.lo = 0;
}

typedef float Row4 __attribute__((ext_vector_type(4)));
typedef const Row4 __attribute__((address_space(1)))* GlobalRow;
typedef const Row4 __attribute__((address_space(3)))* LdsRow;

// Four 16-byte rows of entry i (a node or an instance record, 64 bytes) of an
// array in global memory or, when `lds`, of a TLAS staged in LDS.  Naming the
// address space lets the compiler issue four 16-byte loads instead of generic
// per-dword loads; passing base and index (not a selected pointer) keeps the
// LDS base an LDS address.
template <typename T>
__device__ inline void load_rows(const T* base, uint32_t i, bool lds, float4& a, float4& b, float4& c,
                                 uint4& d) {
    static_assert(sizeof(T) == 64, "64-byte entries");
    Row4 r[4];
    if (lds) {
        LdsRow p = (LdsRow)(base + i);
        r[0] = p[0]; r[1] = p[1]; r[2] = p[2]; r[3] = p[3];
    } else {
        GlobalRow p = (GlobalRow)(base + i);
        r[0] = p[0]; r[1] = p[1]; r[2] = p[2]; r[3] = p[3];
    }
    a = make_float4(r[0].x, r[0].y, r[0].z, r[0].w);
    b = make_float4(r[1].x, r[1].y, r[1].z, r[1].w);
    c = make_float4(r[2].x, r[2].y, r[2].z, r[2].w);
    d = make_uint4(__float_as_uint(r[3].x), __float_as_uint(r[3].y), __float_as_uint(r[3].z),
                   __float_as_uint(r[3].w));
}

// Triangle slot of a BLAS (9 floats, global memory: global loads, not flat).
__device__ inline void load_tri(const float* tris, uint32_t slot, V3& a, V3& b, V3& c) {
    typedef const float __attribute__((address_space(1)))* GlobalFloat;
    const GlobalFloat t = (GlobalFloat)(tris + (size_t)slot * 9);
    a = v3(t[0], t[1], t[2]); b = v3(t[3], t[4], t[5]); c = v3(t[6], t[7], t[8]);
}

// Closest-hit ordering: smaller t, then smaller instance input index, then primitive id.
__device__ inline bool better_hit(float t, uint32_t inst_slot, uint32_t tri_slot, const Best& b,
                                  const InstAux* aux) {
    if (!b.found || t < b.t) return true;
    if (t > b.t) return false;
    uint32_t ia = aux[inst_slot].input_index, ib = aux[b.inst_slot].input_index;
    if (ia != ib) return ia < ib;
    return aux[inst_slot].prims[tri_slot] < aux[b.inst_slot].prims[b.tri_slot];
}

typedef uint32_t Word4 __attribute__((ext_vector_type(4)));
typedef const Word4 __attribute__((address_space(1)))* GlobalWords;
typedef _Float16 Half2 __attribute__((ext_vector_type(2)));

// Bytes 2h and 2h + 1 of w as two FP16 subnormals: the half 0x00qq is q x 2^-24.
template <int H>
__device__ inline Half2 byte_pair(uint32_t w) {
    return __builtin_bit_cast(Half2, __builtin_amdgcn_perm(0u, w, H ? 0x0C030C02u : 0x0C010C00u));
}

// Visit of an 8-wide quantised BLAS node (any-hit): 8 slab tests on the
// decoded child boxes, the hit internal children stacked, then the hit
// triangles tested.
//
// The traversal of large BLASes is bound by VALU issue, most of it this test,
// so the test is shaped for instruction count: no branch per child (empty
// slots are masked at the end; a branch per child also kept the children's
// chains from overlapping and cost four scalar instructions each), two plane
// bytes per v_perm_b32 as FP16 pairs that v_fma_mix_f32 takes as they are
// (instead of one v_cvt_f32_ubyte each), and hit bits from the sign of
// far - near.  Internal and leaf children go in two loops: a wave runs each
// loop as often as its busiest lane needs, and in one loop a lane with a
// triangle made the others wait for it at every position.  VALU instructions
// per node 246 -> 173; frame of the 4K terrain 22.2 -> 20.9 ms (min, max, perm
// and fma_mix issue at 4.4 cycles per wave64 here, add and mul at 2.6 to 2.9, fma at 3.1).
template <typename STACK>
__device__ inline int wide_visit(RayState& r, STACK& st) {
    const GlobalWords p = (GlobalWords)(reinterpret_cast<const Node8*>(r.bnodes) + r.next);
    const Word4 h0 = p[0], h1 = p[1], qa = p[2], qb = p[3], qc = p[4];
    const float ox = __uint_as_float(h0.x), oy = __uint_as_float(h0.y), oz = __uint_as_float(h0.z);
    const int ex = (int)(int8_t)(h0.w & 0xFFu), ey = (int)(int8_t)((h0.w >> 8) & 0xFFu),
              ez = (int)(int8_t)((h0.w >> 16) & 0xFFu);
    const uint32_t nchild = h0.w >> 24;
    // the near and far planes' byte words per axis, chosen once per node by
    // the ray's direction signs (box_hit chooses them per child)
    const bool gx = r.br.inv.x < 0.0f, gy = r.br.inv.y < 0.0f, gz = r.br.inv.z < 0.0f;
    const uint32_t nx[2] = {gx ? qb.z : qa.x, gx ? qb.w : qa.y}, fx[2] = {gx ? qa.x : qb.z, gx ? qa.y : qb.w};
    const uint32_t ny[2] = {gy ? qc.x : qa.z, gy ? qc.y : qa.w}, fy[2] = {gy ? qa.z : qc.x, gy ? qa.w : qc.y};
    const uint32_t nz[2] = {gz ? qc.z : qb.x, gz ? qc.w : qb.y}, fz[2] = {gz ? qb.x : qc.z, gz ? qb.y : qc.w};
    // Distances here are 2^-24 of the ray's (the slab ray is scaled):
    // a child plane o + q x 2^e is met at (o + q x 2^e - ro) x inv =
    // (q x 2^-24) x S + O, with S = 2^(e + 24) x inv (exact: a power-of-two
    // scaling, and the FP16 subnormal holds q x 2^-24 exactly) and
    // O = (o - ro) x inv per node and axis: one fused multiply-add per plane.
    // Its rounding error, like that of decoding the plane first, is a few
    // ulps of the terms, covered as before by the far bound's widening and
    // the child boxes' outward rounding; an infinite reciprocal (a direction
    // component of zero) gives infinite or NaN distances that the max/min
    // ignore or that keep the box, as before.  (On an unscaled ray S overflows
    // for reciprocals from 2^(104 - e), where a near plane at infinity loses
    // boxes that hold the origin.)
    const float Sx = __builtin_ldexpf(r.br.inv.x, ex + 24), Sy = __builtin_ldexpf(r.br.inv.y, ey + 24),
                Sz = __builtin_ldexpf(r.br.inv.z, ez + 24);
    const float Ox = (ox - r.br.o.x) * r.br.inv.x, Oy = (oy - r.br.o.y) * r.br.inv.y,
                Oz = (oz - r.br.o.z) * r.br.inv.z;
    uint32_t miss = 0;   // child k's bit lands at 7 - k
    auto test = [&](float bnx, float bfx, float bny, float bfy, float bnz, float bfz) {
        const float tn = box_near(r.br, __builtin_fmaf(bnx, Sx, Ox), __builtin_fmaf(bny, Sy, Oy),
                                  __builtin_fmaf(bnz, Sz, Oz));
        const float tf = box_far(r.br, __builtin_fmaf(bfx, Sx, Ox), __builtin_fmaf(bfy, Sy, Oy),
                                 __builtin_fmaf(bfz, Sz, Oz));
        // the sign bit of tf - tn, shifted in (no NaN: the range ends are numbers,
        // or the planes of some axis are: see enter_instance)
        miss = __builtin_amdgcn_alignbit(miss, __float_as_uint(tf - tn), 31);
    };
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        auto pair = [&](Half2 a, Half2 b, Half2 c, Half2 d, Half2 e, Half2 f) {
            test((float)a.x, (float)b.x, (float)c.x, (float)d.x, (float)e.x, (float)f.x);
            test((float)a.y, (float)b.y, (float)c.y, (float)d.y, (float)e.y, (float)f.y);
        };
        pair(byte_pair<0>(nx[w]), byte_pair<0>(fx[w]), byte_pair<0>(ny[w]), byte_pair<0>(fy[w]),
             byte_pair<0>(nz[w]), byte_pair<0>(fz[w]));
        pair(byte_pair<1>(nx[w]), byte_pair<1>(fx[w]), byte_pair<1>(ny[w]), byte_pair<1>(fy[w]),
             byte_pair<1>(nz[w]), byte_pair<1>(fz[w]));
    }
    // Bit 7 - k of `inner`: child k is internal (bit 7 of its meta byte); the
    // children of one sort are numbered in slot order, so a child's offset is
    // the number of its sort before it.
    const uint32_t inner =
        __builtin_amdgcn_udot4(h1.w & 0x80808080u, 0x01020408u,
                               __builtin_amdgcn_udot4(h1.z & 0x80808080u, 0x10204080u, 0u, false), false) >> 7;
    const uint32_t used = (0xFF00u >> nchild) & 0xFFu;   // bits 7 .. 8 - nchild
    const uint32_t hit = ~miss & used;
    const uint32_t leaf = ~inner & used;
    r.next = kNone;
    for (uint32_t m = hit & inner; m;) {
        const uint32_t k = 31u - (uint32_t)__builtin_clz(m);
        m &= ~(1u << k);
        const uint32_t child = h1.x + (uint32_t)__popc(inner >> (k + 1));
        if (r.next == kNone) r.next = child;
        else if (!st.push(child)) return kStepOverflow;
    }
    for (uint32_t m = hit & leaf; m;) {
        const uint32_t k = 31u - (uint32_t)__builtin_clz(m);
        m &= ~(1u << k);
        V3 a, b, c;
        load_tri(r.btris, h1.y + (uint32_t)__popc(leaf >> (k + 1)), a, b, c);
        float T, det, U, V, W;
        if (tri_test(r.tr, r.br.o, r.tmin, r.tmax, a, b, c, T, det, U, V, W)) return kStepHit;
    }
    return kStepContinue;
}

// Enters instance `slot`: its object-space ray and BLAS, the root next.  False
// where the ray cannot meet any box of it.
template <bool WIDE>
__device__ inline bool enter_instance(RayState& r, const InstRec* recs, bool recs_lds, uint32_t slot, float thi) {
    float4 w0, w1, w2;
    uint4 pp;
    load_rows(recs, slot, recs_lds, w0, w1, w2, pp);
    float w[12] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w, w2.x, w2.y, w2.z, w2.w};
    V3 oo = xform_point(w, r.wbr.o);
    V3 od = xform_vec(w, r.wd);
    const BoxRay obj = box_setup(oo, od, r.tmin, thi);
    r.tr = tri_setup(od);
    // With a NaN range end, a ray that has no axis of plane distances that are
    // numbers meets no box (its bounds are NaN); wide_visit compares by the sign
    // of a difference, which a NaN does not decide.
    auto numbers = [](float o, float inv) { return fabsf(inv) < INFINITY && o * inv == o * inv; };
    if (WIDE && __builtin_isunordered(r.br.tlo, r.br.thi) && !numbers(oo.x, obj.inv.x) &&
        !numbers(oo.y, obj.inv.y) && !numbers(oo.z, obj.inv.z))
        return false;
    if (WIDE) {   // any-hit: the range is the ray's; an infinite reciprocal stays infinite
        r.br.o = obj.o;
        r.br.inv = v3(obj.inv.x * 0x1p-24f, obj.inv.y * 0x1p-24f, obj.inv.z * 0x1p-24f);
    } else {
        r.br = obj;
    }
    r.bnodes = reinterpret_cast<const Node*>(((uint64_t)pp.y << 32) | pp.x);
    r.btris = reinterpret_cast<const float*>(((uint64_t)pp.w << 32) | pp.z);
    r.inst_slot = slot;
    r.in_blas = true;
    r.next = 0;
    return true;
}

// Visit of a binary node (rows qx, qy, qz, children qc) with slab ray cur: the
// nearer hit child next, the other stacked; hit leaves of a BLAS are tested.
template <bool CLOSEST, typename STACK>
__device__ inline int binary_visit(RayState& r, STACK& st, bool blas, const BoxRay& cur, float4 qx, float4 qy,
                                   float4 qz, uint4 qc, const InstAux* aux, Best* best) {
    float tn0, tn1;
    const bool b0 = box_hit(cur, qx.x, qx.z, qy.x, qy.z, qz.x, qz.z, tn0);
    const bool b1 = box_hit(cur, qx.y, qx.w, qy.y, qy.w, qz.y, qz.w, tn1);
    const bool h0 = (qc.x != kEmpty) & b0;
    const bool h1 = (qc.y != kEmpty) & b1;
    // the hit leaves of a BLAS node (0, 1 or 2 triangles), and its other hit
    // children: the nearer one next, the other stacked
    const bool l0 = h0 && blas && (qc.x & kLeaf), l1 = h1 && blas && (qc.y & kLeaf);
    const bool n0 = h0 && !l0, n1 = h1 && !l1;
    const bool second = n1 && (!n0 || tn1 < tn0);
    r.next = second ? qc.y : (n0 ? qc.x : kNone);
    if (n0 && n1 && !st.push(second ? qc.x : qc.y)) return kStepOverflow;
    // One triangle test in a loop instead of one per child: lanes whose only
    // leaf is child 0 and lanes whose only leaf is child 1 share a pass.
    uint32_t leaf = l0 ? qc.x : qc.y, left = (l0 ? 1u : 0u) + (l1 ? 1u : 0u);
    while (left) {
        const uint32_t slot = leaf & ~kLeaf;
        leaf = qc.y;
        --left;
        V3 a, b, cc;
        load_tri(r.btris, slot, a, b, cc);
        float T, det, U, V, W;
        if (!tri_test(r.tr, r.br.o, r.tmin, r.tmax, a, b, cc, T, det, U, V, W)) continue;
        if (!CLOSEST) return kStepHit;
        float t = __fdiv_rn(T, det);
        if (better_hit(t, r.inst_slot, slot, *best, aux)) {
            best->found = true;
            best->t = t;
            best->inst_slot = r.inst_slot;
            best->tri_slot = slot;
            best->T = T; best->det = det; best->U = U; best->V = V; best->W = W;
            float m = t_margin(t);
            r.br.thi = t + m;
            r.wbr.thi = t + m;
        }
    }
    return kStepContinue;
}

// One node visit of a TLAS-free any-hit ray inside a BLAS (its stack holds
// instance slots and, above r.base, nodes of that BLAS; no sentinel), and the
// next node or instance slot taken from the stack.
template <bool WIDE, typename STACK>
__device__ inline int tlas_free_visit(RayState& r, STACK& st, uint32_t max_steps) {
    if (++r.steps > max_steps) return kStepOverflow;
    int res;
    if (WIDE) {
        res = wide_visit(r, st);
    } else {
        float4 qx, qy, qz;
        uint4 qc;
        load_rows(r.bnodes, r.next, false, qx, qy, qz, qc);
        res = binary_visit<false>(r, st, true, r.br, qx, qy, qz, qc, nullptr, nullptr);
    }
    if (res != kStepContinue || r.next != kNone) return res;
    if (st.sp == 0) return kStepDone;
    r.in_blas = st.sp > r.base;
    r.next = st.pop();
    return kStepContinue;
}

// tlas_lds: tlas_nodes and recs point into LDS (a staged TLAS).
template <bool CLOSEST, bool WIDE = false, typename STACK = Stack>
__device__ inline int ray_step(RayState& r, STACK& st, const Node* tlas_nodes, const InstRec* recs,
                               const InstAux* aux, Best* best, bool tlas_lds = false,
                               uint32_t max_steps = kMaxSteps) {
    if (++r.steps > max_steps) return kStepOverflow;
    if (r.next == kNone) {
        if (st.sp == 0) return kStepDone;
        r.next = st.pop();
        if (r.next == kSentinel) {
            r.in_blas = false;
            r.next = kNone;
            return kStepContinue;
        }
    }
    if (!r.in_blas && (r.next & kLeaf)) {
        if (!st.push(kSentinel)) return kStepOverflow;
        if (!enter_instance<WIDE>(r, recs, tlas_lds, r.next & ~kLeaf, CLOSEST ? best->t : r.tmax)) {
            r.next = kNone;
            r.in_blas = true;   // the sentinel comes next
        }
        return kStepContinue;
    }
    if (WIDE && r.in_blas) return wide_visit(r, st);
    float4 qx, qy, qz;
    uint4 qc;
    load_rows(r.in_blas ? r.bnodes : tlas_nodes, r.next, tlas_lds && !r.in_blas, qx, qy, qz, qc);
    // the ray of the tree being walked, selected per lane (restoring the world
    // ray into a single slot on every return to the TLAS costs more)
    return binary_visit<CLOSEST>(r, st, r.in_blas, r.in_blas ? r.br : r.wbr, qx, qy, qz, qc, aux, best);
}

}  // namespace luz
