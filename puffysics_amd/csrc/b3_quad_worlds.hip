/*
 * b3_quad_worlds.hip - the step on quads of lanes (b3d_quad.h) of the
 * caller's own device-resident B3World structs, in place
 * (b3_batch_step_worlds_gpu): word k of a world is its k-th word, so nothing
 * is transposed or copied, and only the per-step scratch comes from the
 * library's fixed array.
 */
#define B3D_WORD 1
#include "b3d_quad.h"

#include <hip/hip_runtime.h>

#include "b3_engine.h"
#include "b3_engine_internal.h"

using namespace b3d;

namespace {

/* Whether this worker's share of the world's structural checks holds (the
 * checks of b3_engine_create on a world: counts within the capacities, every
 * body and shape index in range). */
B3Q_FN bool quad_world_ok(const QLane& Q) {
    const Lane& L = Q.L;
    const Geometry& g = L.g;
    const uint32_t* w = L.w;
    int nb = ldi(w, H_BODY_COUNT), ns = ldi(w, H_SHAPE_COUNT), nc = ldi(w, H_CONTACT_COUNT), nj = ldi(w, H_JOINT_COUNT);
    if (nb < 0 || nb > g.max_b || ns < 0 || ns > g.max_s || nc < 0 || nc > g.max_c || nj < 0 || nj > g.max_j)
        return false;
    auto in = [](int x, int n) { return x >= 0 && x < n; };
    bool ok = true;
    for (int s = Q.worker; s < ns; s += Q.workers) ok = ok && in(ldi(w, sw(L, s, S_BODY)), nb);
    for (int j = Q.worker; j < nj; j += Q.workers)
        ok = ok && in(ldi(w, jw(L, j, J_BODY_A)), nb) && in(ldi(w, jw(L, j, J_BODY_B)), nb);
    for (int c = Q.worker; c < nc; c += Q.workers)
        ok = ok && in(ldi(w, cw(L, c, C_SHAPE_A)), ns) && in(ldi(w, cw(L, c, C_SHAPE_B)), ns)
            && in(ldi(w, cw(L, c, C_BODY_A)), nb) && in(ldi(w, cw(L, c, C_BODY_B)), nb)
            && in(ldi(w, cw(L, c, C_POINT_COUNT)), kMaxManifold + 1);
    return ok;
}

/* Worlds [0, count) of a chunk: world w at aos + w * stride + offset.  A
 * world that is not selected or not sound is left exactly as it is.  Bound
 * like b3k_step_quad by the worlds' chains; before, each chunk of 896 arm
 * worlds was transposed into tiles, stepped at one lane a world and
 * transposed back: 2.78 ms for 2,000 of them. */
template <int W, int CR, int JR>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(2, 2))) void b3k_step_quad_worlds(uint32_t* aos,
        size_t stride, size_t offset, uint32_t* scratch, size_t tile_words, Geometry g, QuadLayout q, int count,
        float dt, int substeps, const unsigned char* active) {
    extern __shared__ float lds[];
    int* wg = reinterpret_cast<int*>(lds);
    int tile = (int)(blockIdx.x >> 2);
    int slot = (int)(blockIdx.x & 3u) * kQuadCols + (int)((threadIdx.x & 63u) >> 2);
    int w = tile * 64 + slot;
    bool selected = w < count && (!active || active[w]);
    if (__ballot(selected) == 0) return;      /* the same worlds in every wave */
    uint32_t* tile_scratch = scratch + (size_t)tile * tile_words;
    QLane Q = quad_lane(aos + (size_t)(selected ? w : 0) * stride + offset, tile_scratch,
        tile_scratch + q.scratch_tile_words, lds, g, q, slot, W, 0u);
    quad_clear(Q, wg);
    __syncthreads();
    /* the old-contacts-unsorted flag serves for the check: a world that
     * fails it does not step, so nothing reads it as that */
    const int flag = q.hits + hit_words(g);
    if (selected && !quad_world_ok(Q)) lseti(Q, flag, 1);
    __syncthreads();
    Q.L.active = selected && lgeti(Q, flag) == 0;
    __syncthreads();
    quad_step<CR, JR>(Q, dt, substeps, wg, QuadNoLaw{});
}

using WorldsKernel = void (*)(uint32_t*, size_t, size_t, uint32_t*, size_t, Geometry, QuadLayout, int, float, int,
    const unsigned char*);
WorldsKernel worlds_kernel(int max_j) {
    return max_j <= 8 ? b3k_step_quad_worlds<8, 2, 1> : b3k_step_quad_worlds<8, 2, 2>;
}

/* Scratch words of a 64-world tile: its per-lane words and contact records,
 * then its manifold stage. */
size_t worlds_tile_words(const Geometry& g, const QuadLayout& q) {
    size_t stage = (size_t)g.max_s * (size_t)(g.max_s - 1) / 2 * kStageWords;
    return (q.scratch_tile_words + (1 + stage) * kLanes + 3) & ~(size_t)3;
}

}  // namespace

size_t b3i_quad_worlds_tile_words(const Geometry& g) {
    QuadLayout q;
    return quad_layout(g, 8, kCuLdsBytes, 0, &q) ? worlds_tile_words(g, q) : 0;
}

hipError_t b3i_quad_worlds_init() {
    hipError_t err = b3i_lds_limit((const void*)worlds_kernel(8));
    return err == hipSuccess ? b3i_lds_limit((const void*)worlds_kernel(16)) : err;
}

hipError_t b3i_step_quad_worlds(uint32_t* aos, size_t stride, size_t offset, uint32_t* scratch, const Geometry& g,
        int count, float dt, int substeps, const unsigned char* active, hipStream_t stream) {
    QuadLayout q;
    if (!quad_layout(g, 8, kCuLdsBytes, 0, &q)) return hipErrorInvalidValue;
    size_t lds = ((size_t)kQuadWgWords + (size_t)q.words * kQuadCols) * sizeof(float);
    worlds_kernel(g.max_j)<<<(count + 63) / 64 * 4, 512, lds, stream>>>(aos, stride, offset, scratch,
        worlds_tile_words(g, q), g, q, count, dt, substeps, active);
    return hipGetLastError();
}
