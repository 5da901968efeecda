// primary.hip — primary-ray G-buffer producer on gfx950.
//
// The reference rasterises the G-buffer (opaque.vert:21-31, opaque.frag:21-58,
// DeferredRenderer.cpp:254-262); the lighting path's inputs are defined here
// "by primary rays": a persistent closest-hit traversal over the same TLAS,
// writing world position, normalised interpolated vertex normal (through the
// instance's inverse-transpose), and the material of the hit instance.
// Ties in t are broken by (instance input index, primitive id), so the result
// does not depend on traversal order.
#include "closest.hpp"
#include "internal.hpp"

namespace luz {
namespace {

constexpr int kBlock = 256;

// The error latch kCntError is left set until the host reports it.
__global__ void k_clear_tiles(uint32_t* counters) { clear_tile_claims(counters, threadIdx.x); }

// Waves claim 8x8 tiles (lane = pixel of a tile): those that drew cheap tiles
// take more of them.  Bound by the latency of dependent node reads.
__global__ __launch_bounds__(kBlock, 5) void k_primary(TlasView tlas, const InstAux* aux, luzrt_camera cam,
                                                       const luzrt_material* mats, uint32_t nmats,
                                                       luzrt_gbuffer_out out, uint32_t* spill, uint32_t* counters,
                                                       uint32_t chunk) {
    __shared__ uint32_t lds[kShort * kBlock];
    __shared__ float4 staged[kStageFloat4];
    const uint32_t tid = threadIdx.x;
    Stack st;
    st.init(lds + tid, kBlock, spill + (size_t)blockIdx.x * kBlock + tid, gridDim.x * kBlock);
    const TlasView tl = stage_tlas(tlas, staged);
    claim_tiles(counters, ((out.width + 7) / 8) * ((out.height + 7) / 8), chunk, [&](uint32_t tile) {
        primary_tile(tl, aux, cam, mats, nmats, out, tile, st, &counters[kCntError]);
    });
}

}  // namespace

void launch_clear_tiles(hipStream_t st, uint32_t* counters) { k_clear_tiles<<<1, 64, 0, st>>>(counters); }

}  // namespace luz

using namespace luz;

extern "C" luzrt_status luzrt_primary_gbuffer(luzrt_ctx* ctx, const luzrt_tlas* tlas,
                                              const luzrt_camera* cam,
                                              const luzrt_material* materials, uint32_t nmats,
                                              const luzrt_gbuffer_out* out) {
    if (!ctx) return LUZRT_E_INVALID_ARG;
    if (!tlas || !cam || !out || (nmats && !materials) || !out->position || !out->normal ||
        !out->albedo || !out->material || !out->emission)
        return fail(ctx, LUZRT_E_INVALID_ARG, "luzrt_primary_gbuffer: null argument");
    if (out->width == 0 || out->height == 0 || out->width > 16384 || out->height > 16384)
        return fail(ctx, LUZRT_E_LIMIT, "luzrt_primary_gbuffer: size %ux%u outside 1..16384",
                    out->width, out->height);
    luzrt_status s = ensure(ctx, ctx->counters, kCounterBytes);
    if (s != LUZRT_OK) return s;
    if ((s = tlas_acquire(ctx, tlas)) != LUZRT_OK) return s;
    // the material table lives in device memory for the duration of the call
    size_t mbytes = (size_t)(nmats ? nmats : 1) * sizeof(luzrt_material);
    static_assert(sizeof(luzrt_material) == 16, "material layout");
    luzrt_material* dmats = nullptr;
    LUZ_HIP(ctx, hipMallocAsync((void**)&dmats, mbytes, ctx->stream));
    if (nmats)
        LUZ_HIP(ctx, hipMemcpyAsync(dmats, materials, (size_t)nmats * sizeof(luzrt_material),
                                    hipMemcpyHostToDevice, ctx->stream));
    uint32_t groups = (uint32_t)ctx->num_cus * kPrimaryGroupsPerCu;
    if (groups == 0) groups = 1;
    if ((s = ensure(ctx, ctx->spill, (size_t)groups * 256 * kSpill * 4)) != LUZRT_OK) return s;
    uint32_t* counters = (uint32_t*)ctx->counters.ptr;
    stage_begin(ctx, kStagePrimary);
    launch_clear_tiles(ctx->stream, counters);
    const uint32_t ntiles = ((out->width + 7) / 8) * ((out->height + 7) / 8);
    const TlasView view = {tlas->nodes, tlas->recs, tlas_slot_boxes(tlas), tlas->count, false};
    k_primary<<<groups, 256, 0, ctx->stream>>>(view, tlas->aux, *cam, dmats, nmats, *out, (uint32_t*)ctx->spill.ptr,
                                              counters, tile_chunk(ntiles, groups));
    stage_end(ctx, kStagePrimary);
    LUZ_HIP(ctx, hipGetLastError());
    LUZ_HIP(ctx, hipFreeAsync(dmats, ctx->stream));
    return LUZRT_OK;
}
