/*
 * TEST INFRASTRUCTURE ONLY: the LDS layout of the step on quads of lanes, for
 * a test of its regions.
 */
#include "b3d_quad_layout.h"

using namespace b3d;

extern "C" {

/* 0: refused; else 1 and the layout, then the sizes it follows from. */
int quadlayout(unsigned long long sig, int waves, int law_words, int* out) {
    Geometry g;
    size_t world_bytes;
    QuadLayout q;
    if (!geometry_of(sig, &g, &world_bytes) || !quad_layout(g, waves, 163840 * waves / 8, law_words, &q)) return 0;
    const int v[] = {q.hits, q.jkeys, q.last, q.pos, q.level, q.order, q.jlast, q.jlev, q.jgeo, q.jconst, q.heads, q.y,
        q.bounds, q.masks, q.keys, q.clip, q.cw, q.law, q.words, hit_words(g), 4 * kShapeRows, kJGWords, kJCWords,
        quad_body_rows(g), kClipWords, kQuadWgWords, kQuadCols};
    for (int k = 0; k < (int)(sizeof(v) / sizeof(v[0])); k++) out[k] = v[k];
    return 1;
}

}  // extern "C"
