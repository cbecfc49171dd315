/*
 * b3_quad.hip - the step on four lanes of each wave per world (b3d_quad.h)
 * for batches that leave compute units idle at one lane per world, and the
 * step with the built-in force law the same way.
 */
#include "b3d_quad.h"

#include <hip/hip_runtime.h>

#include "b3_engine.h"
#include "b3_engine_internal.h"

using namespace b3d;

namespace {

/* b3k_step on quads.  Bound by each world's chain of solves: at one lane a
 * world a chain of eight hinges (4,096 worlds) took 391 us, 292 of them in
 * 160 levels of joint solves at 1.83 us (a solve's ~400 instructions and
 * ~90 row loads at ~5 cycles each, a wave alone on its SIMD); on quads with
 * the rows in registers 153 us.  W: waves of the workgroup; CR, JR: contacts
 * and joints of a world that a wave keeps in registers (with four contacts
 * the chains took 197 us).  Of the 256 VGPRs that two waves per SIMD allow
 * <8, 2, 1> spills none, <8, 2, 2> and <4, 2, 2> 18, <4, 3, 1> 49 and
 * <4, 1, 4> 61, to private memory. */
template <int W, int CR, int JR, class Law>
__device__ __attribute__((always_inline)) inline void step_quad(uint32_t* live, const uint32_t* snap, uint32_t* scratch,
        uint32_t* stage, size_t stage_tile_words, const Geometry& g, const QuadLayout& q, int count, float dt,
        int substeps, const unsigned char* step_mask, const unsigned char* reset_mask, unsigned int opts, Law law) {
    extern __shared__ float lds[];
    int* wg = reinterpret_cast<int*>(lds);
    int tile = (int)(blockIdx.x >> 2), part = (int)(blockIdx.x & 3u);
    int slot = part * kQuadCols + (int)((threadIdx.x & 63u) >> 2);
    if (reset_mask) {
        uint64_t mine = ((1ull << kQuadCols) - 1) << (part * kQuadCols);
        restore_tile(live, snap, g, count, reset_mask, tile, (int)(threadIdx.x >> 6), W, mine);
    }
    int w = tile * 64 + slot;
    bool stepping = w < count && (!step_mask || step_mask[w]);
    /* every wave holds the same worlds, so the workgroup returns as a whole */
    if (!(dt > 0.0f) || __ballot(stepping) == 0) return;
    QLane Q = quad_lane(live + (size_t)tile * g.world_words * kLanes + slot,
        scratch + (size_t)tile * q.scratch_tile_words, stage + (size_t)tile * stage_tile_words, lds, g, q, slot, W, opts);
    Q.L.active = stepping;
    quad_clear(Q, wg);
    __syncthreads();
    if constexpr (Law::kWords > 0) {
        if (law.masses) law.masses += (size_t)w * g.max_b;
    }
    quad_step<CR, JR>(Q, dt, substeps, wg, law);
}

template <int W, int CR, int JR>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(2, 2))) void b3k_step_quad(uint32_t* live,
        const uint32_t* snap, uint32_t* scratch, uint32_t* stage, size_t stage_tile_words, Geometry g, QuadLayout q,
        int count, float dt, int substeps, const unsigned char* step_mask, const unsigned char* reset_mask,
        unsigned int opts) {
    step_quad<W, CR, JR>(live, snap, scratch, stage, stage_tile_words, g, q, count, dt, substeps, step_mask, reset_mask,
        opts, QuadNoLaw{});
}

/* The step with gravity between each world's bodies.  At one lane a world
 * the pair loop's loads and stores went through memory, 136 pairs in turn a
 * substep for 17 bodies (4.06 ms for 1,000 arm worlds); here a worker sums
 * one body's pairs from LDS. */
template <int W, int CR, int JR>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(2, 2))) void b3k_step_quad_gravity(
        uint32_t* live, const uint32_t* snap, uint32_t* scratch, uint32_t* stage, size_t stage_tile_words, Geometry g,
        QuadLayout q, int count, float dt, int substeps, const unsigned char* step_mask,
        const unsigned char* reset_mask, unsigned int opts, B3GravityLaw law, const float* masses) {
    step_quad<W, CR, JR>(live, snap, scratch, stage, stage_tile_words, g, q, count, dt, substeps, step_mask, reset_mask,
        opts, QuadGravity{law.gravity, law.softening, masses});
}

using QuadKernel = void (*)(uint32_t*, const uint32_t*, uint32_t*, uint32_t*, size_t, Geometry, QuadLayout, int, float,
    int, const unsigned char*, const unsigned char*, unsigned int);
QuadKernel quad_kernel(int waves, int max_j) {
    if (waves == 8) return max_j <= 8 ? b3k_step_quad<8, 2, 1> : b3k_step_quad<8, 2, 2>;
    return max_j <= 4 ? b3k_step_quad<4, 3, 1> : (max_j <= 8 ? b3k_step_quad<4, 2, 2> : b3k_step_quad<4, 1, 4>);
}
using QuadGravityKernel = void (*)(uint32_t*, const uint32_t*, uint32_t*, uint32_t*, size_t, Geometry, QuadLayout, int,
    float, int, const unsigned char*, const unsigned char*, unsigned int, B3GravityLaw, const float*);
QuadGravityKernel quad_gravity_kernel(int waves, int max_j) {
    if (waves == 8) return max_j <= 8 ? b3k_step_quad_gravity<8, 2, 1> : b3k_step_quad_gravity<8, 2, 2>;
    return max_j <= 8 ? b3k_step_quad_gravity<4, 2, 2> : b3k_step_quad_gravity<4, 1, 4>;
}

/* A workgroup of eight waves has the CU's LDS to itself, one of four half. */
size_t quad_lds_bytes(int waves) { return kCuLdsBytes * waves / 8; }
size_t quad_lds_of(const QuadLayout& q) {
    return ((size_t)kQuadWgWords + (size_t)q.words * kQuadCols) * sizeof(float);
}

}  // namespace

bool b3i_quad_fit(const Geometry& g, int waves, size_t* scratch_tile_words) {
    QuadLayout q;
    if (!quad_layout(g, waves, quad_lds_bytes(waves), 0, &q)) return false;
    *scratch_tile_words = q.scratch_tile_words;
    return true;
}

hipError_t b3i_quad_init() {
    for (int waves = 4; waves <= 8; waves += 4)
        for (int max_j = 4; max_j <= 16; max_j += 4) {
            hipError_t err = b3i_lds_limit((const void*)quad_kernel(waves, max_j));
            if (err == hipSuccess) err = b3i_lds_limit((const void*)quad_gravity_kernel(waves, max_j));
            if (err != hipSuccess) return err;
        }
    return hipSuccess;
}

hipError_t b3i_step_quad(B3Engine* e, float dt, int substeps, const unsigned char* step_mask,
        const unsigned char* reset_mask, hipStream_t stream) {
    QuadLayout q;
    if (!quad_layout(e->g, e->quad_waves, quad_lds_bytes(e->quad_waves), 0, &q)) return hipErrorInvalidValue;
    QuadKernel kernel = quad_kernel(e->quad_waves, e->g.max_j);
    kernel<<<e->tiles * 4, 64 * e->quad_waves, quad_lds_of(q), stream>>>(e->live, e->snap, e->scratch, e->pair_stage,
        e->stage_tile_words, e->g, q, e->count, dt, substeps, step_mask, reset_mask, e->options);
    return hipGetLastError();
}

bool b3i_step_quad_gravity(B3Engine* e, float dt, int substeps, const unsigned char* step_mask,
        const unsigned char* reset_mask, B3GravityLaw law, const float* masses, hipStream_t stream, hipError_t* err) {
    QuadLayout q;
    if (!e->quad_waves
            || !quad_layout(e->g, e->quad_waves, quad_lds_bytes(e->quad_waves), QuadGravity::kWords, &q))
        return false;
    QuadGravityKernel kernel = quad_gravity_kernel(e->quad_waves, e->g.max_j);
    kernel<<<e->tiles * 4, 64 * e->quad_waves, quad_lds_of(q), stream>>>(e->live, e->snap, e->scratch, e->pair_stage,
        e->stage_tile_words, e->g, q, e->count, dt, substeps, step_mask, reset_mask, e->options, law, masses);
    *err = hipGetLastError();
    return true;
}
