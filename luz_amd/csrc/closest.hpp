// closest.hpp — closest-hit launches over 8x8 tiles of rays (gfx950): primary
// rays (primary.hip, batch.hip) and shadow-map texels (shadowmap.hip).
//
// The 64 rays of a tile are one beam.  With at most kMaxCullInst instances no
// TLAS node is visited: the wave tests the slots' padded world boxes against
// the beam (lane = slot), each lane then its own ray against the few boxes
// left, and its nearest one is entered first.  A ray that leaves an instance
// enters its next one at once: where such rays wait for each other, as in the
// culled any-hit traversal, the longest rays of a tile get longer (shadow maps of
// 1024 texels: 5.0 ms against 4.6).  Primary rays 1280x720 297 -> 280 us, shadow
// maps 6.20 -> 4.55 ms against the walk from the TLAS root.
#pragma once
#include "cull.hpp"

namespace luz {

// Calls tile(i) for tiles 0 .. ntiles - 1 of a persistent launch, `chunk`
// consecutive ones per claim: a wave's first chunk is the one of its number,
// the rest are claimed from the counter of its workgroup's segment (one of
// kClaimSegments, workgroups in turn, so a segment's waves share an XCD), which
// deals chunks s, s + 8, s + 16, ... of those left.  A device-scope atomic on one
// address takes about 21 ns whoever asks, and one counter bounded whole
// launches: 14,400 tiles of 1280x720 and 5,120 waves that find none left took
// 420 us (297 with eight), the 12 frames of a batch 1910 us (970).  A segment's
// waves do not look at the other counters: neighbouring chunks belong to
// different segments, so all eight end together, and the polls would queue again.
template <typename F>
__device__ inline void claim_tiles(uint32_t* counters, uint32_t ntiles, uint32_t chunk, F&& tile) {
    const uint32_t lane = threadIdx.x & 63u, nseg = min(kClaimSegments, gridDim.x);
    const uint32_t seg = blockIdx.x % nseg, waves = gridDim.x * (blockDim.x >> 6);
    const uint32_t nchunks = (uint32_t)(((uint64_t)ntiles + chunk - 1) / chunk);
    uint32_t c = (threadIdx.x >> 6) * gridDim.x + blockIdx.x;
    while (c < nchunks) {
        const uint32_t begin = c * chunk, end = min(begin + chunk, ntiles);
        for (uint32_t i = begin; i < end; ++i) tile(i);
        if (waves >= nchunks) break;
        uint32_t got = 0;
        if (lane == 0) got = atomicAdd(&counters[kTileBase + seg * kClaimStride], 1u);
        const uint64_t next = (uint64_t)__shfl(got, 0) * nseg + seg + waves;
        if (next >= nchunks) break;
        c = (uint32_t)__builtin_amdgcn_readfirstlane((int)next);
    }
}

// The TLAS of a closest-hit launch: nodes and instance records, and the slots'
// padded world boxes (6 floats each).  `lds`: records and boxes point into LDS.
struct TlasView {
    const Node* nodes;
    const InstRec* recs;
    const float* slot_box;
    uint32_t ninst;
    bool lds;
};

// Staging of a single-scene launch's records and boxes (all threads of the
// workgroup): 11 KB, which with the 16 KB of stacks leaves five workgroups per CU.
constexpr uint32_t kStageFloat4 = kMaxCullInst * 4 + kMaxCullInst * 6 / 4;
__device__ inline TlasView stage_tlas(const TlasView& v, float4* lds) {
    if (v.ninst > kMaxCullInst) return v;
    const float4* gr = reinterpret_cast<const float4*>(v.recs);
    float* boxes = reinterpret_cast<float*>(lds + kMaxCullInst * 4);
    for (uint32_t i = threadIdx.x; i < v.ninst * 4; i += blockDim.x) lds[i] = gr[i];
    for (uint32_t i = threadIdx.x; i < v.ninst * 6; i += blockDim.x) boxes[i] = v.slot_box[i];
    __syncthreads();
    return TlasView{v.nodes, reinterpret_cast<const InstRec*>(lds), boxes, v.ninst, true};
}

__device__ inline void load_slot_box(const TlasView& v, uint32_t slot, float b[6]) {
    if (v.lds) {
        typedef const float __attribute__((address_space(3)))* LdsFloat;
        const LdsFloat p = (LdsFloat)(v.slot_box + slot * 6);
        for (int k = 0; k < 6; ++k) b[k] = p[k];
    } else {
        typedef const float __attribute__((address_space(1)))* GlobalFloat;
        const GlobalFloat p = (GlobalFloat)(v.slot_box + (size_t)slot * 6);
        for (int k = 0; k < 6; ++k) b[k] = p[k];
    }
}
__device__ inline bool slot_box_hit(const BoxRay& r, const float b[6], float& tn) {
    return box_hit(r, b[0], b[3], b[1], b[4], b[2], b[5], tn);
}

// The beam of a wave's rays: the bounds of their origins and of their
// reciprocal directions, per axis.  An axis on which the directions differ in
// sign or a bound is not finite bounds nothing.
struct Beam {
    float o0[3], o1[3], i0[3], i1[3];
    bool use[3], neg[3];
};
__device__ inline Beam beam_of(const BoxRay& r) {
    const float v[6] = {r.o.x, r.o.y, r.o.z, r.inv.x, r.inv.y, r.inv.z};
    float lo[6], hi[6];
    wave_bounds(v, lo, hi);
    Beam b;
    for (int k = 0; k < 3; ++k) {
        const float a = lo[3 + k], c = hi[3 + k];
        b.neg[k] = c < 0.0f;
        b.use[k] = (a > 0.0f || c < 0.0f) && isfinite(a) && isfinite(c) && isfinite(lo[k]) && isfinite(hi[k]);
        // on a negative axis everything is mirrored
        b.o0[k] = b.neg[k] ? -hi[k] : lo[k];
        b.o1[k] = b.neg[k] ? -lo[k] : hi[k];
        b.i0[k] = b.neg[k] ? -c : a;
        b.i1[k] = b.neg[k] ? -a : c;
    }
    return b;
}
// Can any ray of the beam, within [tlo, thi], meet the box widened by the
// margin of cull_group's bounds?  The earliest entry and the latest exit of any
// origin and direction of the beam, axis by axis.
__device__ inline bool beam_meets_box(const Beam& m, const float box[6], float tlo, float thi) {
    float tn = tlo, tf = thi;
    for (int k = 0; k < 3; ++k) {
        if (!m.use[k]) continue;
        const float lo = m.neg[k] ? -box[3 + k] : box[k], hi = m.neg[k] ? -box[k] : box[3 + k];
        const float mag = fmaxf(fmaxf(fabsf(lo), fabsf(hi)), fmaxf(fabsf(m.o0[k]), fabsf(m.o1[k])));
        const float w = 1e-3f + 2e-5f * mag;
        const float a = (lo - w) - m.o1[k], b = (hi + w) - m.o0[k];
        tn = fmaxf(tn, a * (a >= 0.0f ? m.i0[k] : m.i1[k]));
        tf = fminf(tf, b * (b >= 0.0f ? m.i1[k] : m.i0[k]));
    }
    return !(tn > tf + 1e-5f * (fabsf(tn) + fabsf(tf)));
}

// The closest hits of a wave's 64 rays (all lanes active; tmin and tmax the
// wave's).  Ties in t go by (instance input index, primitive id), so the order
// in which instances are entered does not show.
template <typename STACK>
__device__ inline void closest_hits(const TlasView& tl, const InstAux* aux, V3 o, V3 d, float tmin, float tmax,
                                    STACK& st, uint32_t* error_flag, Best& best) {
    RayState r;
    ray_begin(r, st, o, d, tmin, tmax);
    if (tl.ninst > kMaxCullInst) {
        for (;;) {
            const int res = ray_step<true>(r, st, tl.nodes, tl.recs, aux, &best);
            if (res == kStepDone || (res == kStepContinue && r.next == kNone && st.sp == 0)) return;
            if (res == kStepOverflow) { atomicOr(error_flag, 1u); return; }
        }
    }
    const uint32_t lane = threadIdx.x & 63u;
    const Beam beam = beam_of(r.wbr);
    uint64_t mine[kCandWords] = {};   // slots whose boxes this lane's ray meets and has yet to enter
    uint32_t first = kNone;           // the nearest of them
    float first_t = 0.0f;
    for (uint32_t w = 0; w < kCandWords && w * 64 < tl.ninst; ++w) {
        const uint32_t slot = w * 64 + lane;
        bool meets = false;
        if (slot < tl.ninst) {
            float b[6];
            load_slot_box(tl, slot, b);
            meets = beam_meets_box(beam, b, r.wbr.tlo, r.wbr.thi);
        }
        uint64_t todo = __ballot(meets);
        while (todo) {
            const uint32_t s = (uint32_t)__builtin_ctzll(todo);
            todo &= todo - 1;
            float b[6], tn;
            load_slot_box(tl, w * 64 + s, b);
            if (slot_box_hit(r.wbr, b, tn)) {
                mine[w] |= 1ull << s;
                if (first == kNone || tn < first_t) {
                    first = w * 64 + s;
                    first_t = tn;
                }
            }
        }
    }
    bool waiting = first != kNone;   // before instance r.next
    r.next = first;
    if (waiting) mine[first >> 6] &= ~(1ull << (first & 63u));
    for (;;) {
        if (__ballot(waiting || r.in_blas) == 0ull) return;
        if (waiting) {
            enter_instance<false>(r, tl.recs, tl.lds, r.next, best.t);
            waiting = false;
        }
        if (!r.in_blas) continue;
        int res = kStepOverflow;
        if (++r.steps <= kMaxSteps) {
            float4 qx, qy, qz;
            uint4 qc;
            load_rows(r.bnodes, r.next, false, qx, qy, qz, qc);
            res = binary_visit<true>(r, st, true, r.br, qx, qy, qz, qc, aux, &best);
        }
        if (res == kStepOverflow) {
            atomicOr(error_flag, 1u);
            r.in_blas = false;
            mine[0] = mine[1] = 0;
        } else if (r.next == kNone) {
            if (st.sp) {
                r.next = st.pop();
            } else {
                r.in_blas = false;
                while (mine[0] | mine[1]) {   // the next one that the hit so far does not hide
                    const uint32_t w = mine[0] ? 0u : 1u, s = (uint32_t)__builtin_ctzll(w ? mine[1] : mine[0]);
                    if (w) mine[1] &= mine[1] - 1;
                    else mine[0] &= mine[0] - 1;
                    float b[6], tn;
                    load_slot_box(tl, w * 64 + s, b);
                    if (slot_box_hit(r.wbr, b, tn)) {
                        waiting = true;
                        r.next = w * 64 + s;
                        break;
                    }
                }
            }
        }
    }
}

// G-buffer texels of 8x8 tile `tile` of an image (lane = pixel) by primary rays;
// lanes outside the image repeat its last column or row and write nothing.
template <typename STACK>
__device__ inline void primary_tile(const TlasView& tl, const InstAux* aux, const luzrt_camera& cam,
                                    const luzrt_material* mats, uint32_t nmats, const luzrt_gbuffer_out& out,
                                    uint32_t tile, STACK& st, uint32_t* error_flag) {
    const uint32_t lane = threadIdx.x & 63u, W = out.width, H = out.height, tiles_x = (W + 7) / 8;
    const uint32_t x = (tile % tiles_x) * 8 + (lane & 7u), y = (tile / tiles_x) * 8 + (lane >> 3);
    Best best;
    best.found = false;
    best.t = cam.tmax;
    const V3 d = primary_dir(cam, min(x, W - 1), min(y, H - 1), W, H);
    if (tl.ninst)
        closest_hits(tl, aux, v3(cam.eye[0], cam.eye[1], cam.eye[2]), d, cam.tmin, cam.tmax, st, error_flag, best);
    if (x < W && y < H) primary_texel(cam, d, best, aux, mats, nmats, out, x, y);
}

}  // namespace luz
