/*
 * b3_art_world.hip - b3_step with articulated contacts (b3_art.hip), one
 * world to a wave, for batches that leave most of the chip idle at 64.
 *
 * Only the worlds whose contacts go through their joint trees are stepped
 * here, from where b3k_step_art leaves them: a wave has nothing to share out
 * in any other world, and 64 of those step together there.
 *
 * The lane code is built here with one world to a tile (as the CPU step
 * is): a world's words, workspace and rows are contiguous.  A workgroup of
 * one wave copies its world out of the tiles, steps it and writes what a
 * step can change back.  The workspace and the velocities are in LDS; the
 * world stays in global memory, where its lines are in the L1 and L2 (in
 * LDS, 52 KB a world, three worlds fit a CU: 14.1 ms for 1,000 arm worlds,
 * 6.3 for 300, where the whole step was here: 5.6 for 1,000).
 */
#define B3D_LANES 1
#define B3D_ART_WAVE 1
#include "b3d_art.h"

#include <hip/hip_runtime.h>

#include "b3_engine.h"
#include "b3_engine_internal.h"

using namespace b3d;

namespace {

/* Worlds of one 64-byte sector of the tiles' rows: they are stepped on one
 * XCD, whose L2 then reads each sector once for the sixteen copies. */
constexpr int kGroup = 16, kXcds = 8;

/* LDS words: the workspace, the rows (each from a multiple of four words),
 * then what lane 0 found of its tree. */
B3D_FN int vel_word(const Geometry& g) { return (art_ws_words(g.max_b) + 3) & ~3; }
B3D_FN int tree_word(const Geometry& g) { return vel_word(g) + ((lds_rows(g) + 3) & ~3); }
size_t lds_bytes_of(const Geometry& g) { return (size_t)(tree_word(g) + 4) * sizeof(uint32_t); }

/* Words [lo, hi) of the wave's world, to its column of the tile.  A word
 * that has not changed is written again: the row is in the L2 and reading it
 * to compare costs a round trip. */
B3D_FN void put_words(const uint32_t* world, uint32_t* column, int lo, int hi) {
    for (int k = lo + (int)threadIdx.x; k < hi; k += 64) column[(size_t)k * 64] = world[k];
}

/* The rest of step_world_art on a wave, for a world that b3k_step_art has
 * handed over: its contacts are found and prepared, and its trees build.  The
 * parts the ordinary step shares run on lane 0, the articulated passes on all
 * lanes (B3D_ART_WAVE).  Bound by the chain of ~1,000 impulse responses a
 * step (every contact point, twice a substep), each of which goes through
 * every link: 32 ms for the 17 links of an arm world with 64 worlds to a
 * wave, whose lanes hold different links; 18 ms with a world to itself on one
 * lane; 4.3 with a link to a lane, the links outside the trees then in one
 * pass (1,000 worlds 4.9). */
__device__ inline void step_world_art_wave(const Lane& L, float* ws, int* tree, float dt, int substeps) {
    bool one = threadIdx.x == 0;
    ArtParams P = art_params(L, dt, substeps);
    ArtWs A = art_ws_of(L, ws);
    if (one) {
        body_prepass(L, P.h);
        prepare_joints(L, P.h);
        art_build(L, A);
        tree[0] = A.n_links;
        tree[1] = A.n_tree;
    }
    __syncthreads();
    A.n_links = tree[0];
    A.n_tree = tree[1];
    art_warm_start(L, A);
    __syncthreads();
    if (one) {
        warm_start_joints(L);
        joint_geometry(L);
    }
    for (int s = 0; s < P.subs; s++) {
        if (one) integrate_velocities(L);
        __syncthreads();
        art_solve_contacts(L, A, P.inv_h, P.contact_speed, 1);
        __syncthreads();
        if (one) {
            solve_joints(L, P.h, P.inv_h, 1);
            integrate_positions(L, P.h, P.inv_dt);
            delta_geometry(L);
        }
        __syncthreads();
        art_solve_contacts(L, A, P.inv_h, P.contact_speed, 0);
        __syncthreads();
        if (one) {
            solve_joints(L, P.h, P.inv_h, 0);
            wrow_restitution(L, P.rest_threshold);
        }
    }
    if (one) {
        finalize(L);
        vel_store(L);
    }
}

/* The worlds that b3k_step_art<false> handed over, one to a workgroup; at
 * most 256 VGPRs, so that two waves share a SIMD (4,000 arm worlds 20.0 ->
 * 11.4 ms). */
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2))) void b3k_step_art_world(uint32_t* live,
        uint32_t* worlds, uint32_t* scratch, Geometry g, int count, float dt, int substeps,
        const unsigned char* handed, unsigned int opts) {
    extern __shared__ uint32_t lds[];
    int turn = (int)blockIdx.x / kXcds;
    int w = (turn / kGroup * kXcds + (int)blockIdx.x % kXcds) * kGroup + turn % kGroup;
    if (w >= count || !handed[w]) return;
    int tile = w / 64, slot = w % 64;
    uint32_t* column = live + (size_t)tile * g.world_words * 64 + slot;
    uint32_t* world = worlds + (size_t)w * g.world_words;
    for (int k0 = (int)threadIdx.x; k0 < g.world_words; k0 += 64 * 16) {
        uint32_t v[16];
#pragma unroll
        for (int i = 0; i < 16; i++)
            if (k0 + 64 * i < g.world_words) v[i] = column[(size_t)(k0 + 64 * i) * 64];
#pragma unroll
        for (int i = 0; i < 16; i++)
            if (k0 + 64 * i < g.world_words) world[k0 + 64 * i] = v[i];
    }
    __syncthreads();
    float* rows = reinterpret_cast<float*>(lds);
    Lane L = lane_view(world, scratch, rows + vel_word(g), g, 0, 0, opts, w);
    step_world_art_wave(L, rows, reinterpret_cast<int*>(lds) + tree_word(g), dt, substeps);
    __syncthreads();
    /* the step writes no shape, and no contact past the new count */
    int contacts = (int)world[H_CONTACT_COUNT];
    put_words(world, column, 0, g.so);
    put_words(world, column, g.co, g.co + contacts * kContactWords);
    put_words(world, column, g.jo, g.jo + g.max_j * kJointWords);
}

}  // namespace

int b3i_art_worlds_per_cu(const Geometry& g) {
    size_t fit = kCuLdsBytes / lds_bytes_of(g);
    return fit < 8 ? (int)fit : 8;
}

hipError_t b3i_art_world_init() {
    return b3i_lds_limit((const void*)b3k_step_art_world);
}

hipError_t b3i_step_art_world(B3Engine* e, float dt, int substeps, const unsigned char* handed, hipStream_t stream) {
    /* the engine's geometry with this file's one-world scratch tiles: 64 of
     * them are the words of one of the engine's */
    Geometry g;
    size_t world_bytes;
    if (!geometry_of(e->sig, &g, &world_bytes)) return hipErrorInvalidValue;
    int groups = (e->count + kGroup - 1) / kGroup;
    int grid = (groups + kXcds - 1) / kXcds * kXcds * kGroup;
    b3k_step_art_world<<<grid, 64, lds_bytes_of(g), stream>>>(e->live, e->art_worlds, e->scratch, g, e->count, dt,
        substeps, handed, e->options);
    return hipGetLastError();
}
