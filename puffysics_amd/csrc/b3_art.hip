/*
 * b3_art.hip - the engine's steps of the reference's B3_ART_CONTACTS=1
 * build (B3_ENGINE_ART_CONTACTS): b3_step with articulation-aware contacts,
 * and b3_art_step, the reduced-coordinate integrator.
 *
 * Same launch as b3k_step (one wave64 workgroup per tile of 64 worlds, one
 * world per lane, optional fused masked restore).  Of smaller batches the
 * first hands the worlds whose contacts go through their joint trees to a
 * wave each (b3_art_world.hip).  Each lane also owns a
 * workspace of art_ws_words(max_bodies) words, word-transposed across the
 * tile like the worlds, for its world's joint tree (b3d_art.h).
 */
#include <hip/hip_runtime.h>

#include <math.h>

#include "b3_engine.h"
#include "b3_engine_internal.h"
#include "b3d_art.h"

using namespace b3d;

namespace {

/* Reduced: b3_art_step (the reduced-coordinate integrator); otherwise
 * b3_step with articulated contacts. */
template <bool Reduced>
__global__ __launch_bounds__(64) void b3k_step_art(uint32_t* live, const uint32_t* snap, uint32_t* scratch,
        float* art_ws, Geometry g, int count, float dt, int substeps, const unsigned char* step_mask,
        const unsigned char* reset_mask, unsigned int opts, unsigned char* handed) {
    extern __shared__ float vel_rows[];
    if (reset_mask) {
        restore_tile(live, snap, g, count, reset_mask, blockIdx.x, 0, 1);
        __syncthreads();
    }
    int tile = blockIdx.x;
    int lane = threadIdx.x;
    int w = tile * 64 + lane;
    if (w >= count) return;
    if (step_mask && !step_mask[w]) {
        if (handed) handed[w] = 0;
        return;
    }
    float* ws = art_ws + (size_t)tile * art_ws_words(g.max_b) * 64 + lane;
    Lane L = lane_view(live, scratch, vel_rows, g, tile, lane, opts);
    if (Reduced) step_world_art_reduced(L, ws, dt, substeps);
    else step_world_art(L, ws, dt, substeps, handed ? handed + w : nullptr);
}

}  // namespace

/* The largest batch whose articulated worlds take a wave each
 * (b3_art_world.hip): this many turns of as many such waves as the chip
 * holds.  A turn takes about as long as its longest world, so the time grows
 * by turns; 64 to a wave, every lane waits for every other's rows, but 1,024
 * tiles are one turn.  Measured at the rule's edge, ms a vector step, one ->
 * 64 to a wave: the arm's 17 bodies (eight waves a CU) 38.7 at 16,384 worlds,
 * 49.2 at 17,000; twice the bodies (five) 216 at 10,240, 409 at 10,304; four
 * times (two) 903 at 4,096, 2,099 at 4,160.  Worlds that do not go through
 * trees never leave the 64: at 16,384 chains that touch nothing take 0.84,
 * stacks 0.47, bins 4.2 (a wave each, they took 9.7, 4.2 and 38.8). */
constexpr int kArtWorldTurns = 8;
static bool world_per_wave(const B3Engine* e, int cus) {
    return e->count <= kArtWorldTurns * cus * b3i_art_worlds_per_cu(e->g);
}

/* The articulated steps' device memory and launch limits: called by
 * b3_engine_set_options when the option is first turned on. */
hipError_t b3i_art_init(B3Engine* e) {
    hipError_t err = b3i_lds_limit((const void*)b3k_step_art<false>);
    if (err == hipSuccess) err = b3i_lds_limit((const void*)b3k_step_art<true>);
    if (err == hipSuccess) err = b3i_art_world_init();
    if (err != hipSuccess) return err;
    if (e->tiles == 0) return hipSuccess;
    if (!e->art_ws) {
        size_t bytes = (size_t)e->tiles * art_ws_words(e->g.max_b) * 64 * sizeof(float);
        if ((err = hipMalloc((void**)&e->art_ws, bytes)) != hipSuccess) return err;
    }
    int cus = 0;
    if ((err = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, e->device)) != hipSuccess) return err;
    if (!e->art_worlds && world_per_wave(e, cus)) {
        /* where there is no room for it, the batch steps 64 worlds to a wave */
        err = hipMalloc((void**)&e->art_worlds, (size_t)e->count * (e->world_bytes + 1));
        if (err == hipErrorOutOfMemory) {
            (void)hipGetLastError();
            e->art_worlds = nullptr;
            err = hipSuccess;
        }
    }
    return err;
}

hipError_t b3i_step_art(B3Engine* e, float dt, int substeps, const unsigned char* step_mask,
        const unsigned char* reset_mask, hipStream_t stream) {
    unsigned char* handed = e->art_worlds ? (unsigned char*)e->art_worlds + (size_t)e->count * e->world_bytes : nullptr;
    b3k_step_art<false><<<e->tiles, 64, e->lds_bytes, stream>>>(e->live, e->snap, e->scratch, e->art_ws, e->g,
        e->count, dt, substeps, step_mask, reset_mask, e->options, handed);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess || !handed) return err;
    return b3i_step_art_world(e, dt, substeps, handed, stream);
}

extern "C" hipError_t b3_batch_art_step_gpu(B3Engine* e, float dt, int substeps, const unsigned char* step_mask,
        const unsigned char* reset_mask, hipStream_t stream) {
    if (!e || !isfinite(dt) || dt < 0.0f || substeps < 1) return hipErrorInvalidValue;
    if (!(e->options & B3_ENGINE_ART_CONTACTS)) return hipErrorNotSupported;
    if (e->count == 0) return hipSuccess;
    hipError_t err = on_device(e);
    if (err != hipSuccess) return err;
    if (dt == 0.0f) return reset_mask ? b3_batch_restore_gpu(e, reset_mask, stream) : hipSuccess;
    b3k_step_art<true><<<e->tiles, 64, e->lds_bytes, stream>>>(e->live, e->snap, e->scratch, e->art_ws, e->g,
        e->count, dt, substeps, step_mask, reset_mask, e->options, nullptr);
    return hipGetLastError();
}
