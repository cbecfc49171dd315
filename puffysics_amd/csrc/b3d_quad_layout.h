/*
 * b3d_quad_layout.h - the LDS and scratch layout of the step on quads of lanes
 * (b3d_quad.h).  Host and device.  Include before any other header of the
 * engine.
 */
#ifndef PUFFYSICS_AMD_B3D_QUAD_LAYOUT_H
#define PUFFYSICS_AMD_B3D_QUAD_LAYOUT_H

#define B3D_QUAD 1
#define B3D_ROW 16
#include "b3d_lane.h"

namespace b3d {

/* ---- the workgroup's LDS, per world, in words (rows of B3D_ROW) ----
 * Region X, while contacts are generated: the shape records, the candidates'
 * hit bits and the old-contacts-unsorted flag, the joint keys; afterwards
 * the contact levels, the joint levels and the joints' geometry.  Past it,
 * the new contacts' heads.  Region Y, while contacts are generated: shape
 * bounds, overlap masks, old contact keys and the colliding workers' clip
 * rows; afterwards the bodies' rows (quad_body_rows). */
constexpr int kQuadCols = B3D_ROW;
/* words of the workgroup (not per world) at the start of LDS */
constexpr int WG_LEVELS = 0, WG_JLEVELS = 1, WG_JOINTS = 2, WG_REST = 3, kQuadWgWords = 16;
/* joint geometry quads (struct JGeo): a vector and a scalar each; a weld's
 * angular error is in JG_PY */
enum { JG_RA_TW, JG_RB_RELX, JG_PSEP_RELY, JG_PX_KXX, JG_PY_KXY, JG_K0_KYY, JG_K1_KINV, JG_K2, kJGQuads };
constexpr int kJGWords = 4 * kJGQuads;
/* what a joint's geometry reads besides the delta poses, fixed for the step */
constexpr int JC_AB = 0, JC_INFO = 1, JC_QA = 2, JC_QB = 6, JC_PA = 10, JC_PB = 13, JC_DC = 16, JC_MA = 19, JC_MB = 20,
              JC_IA = 21, JC_IB = 30, kJCWords = 39;
/* contact head: body a | body b << 8 | points << 16 | CF_* flags << 20 */
struct QuadLayout {
    int hits, jkeys;                    /* X, contact generation (the shape records are at 0) */
    int last, pos, level, order;        /* X, contact levels */
    int jlast, jlev, jgeo, jconst;      /* X, joints */
    int heads;
    int y;                              /* region Y: the bodies' rows */
    int bounds, masks, keys, clip, cw;  /* Y, contact generation; cw workers collide */
    int law;                            /* rows of a force law, past everything else */
    int waves;                          /* of the workgroup */
    int words;                          /* in all, per world */
    size_t scratch_tile_words;          /* HBM, per tile: the per-lane words, then the contact records */
};
/* contact records in HBM, world after world, contact after contact */
constexpr int kQRecQuads = 26, kQRecWords = 4 * kQRecQuads;
enum { QR_N, QR_T1, QR_CA, QR_CB, QR_IA, QR_IB = QR_IA + 3, QR_ROLL = QR_IB + 3, QR_FI, QR_NMASS, QR_NI, QR_TN, QR_LEVER,
       QR_SEP, QR_RV, QR_RA, QR_RB = QR_RA + 4 };
static_assert(QR_RB + 4 == kQRecQuads, "contact record quads");

/* The layout of a capacity set for workgroups of `waves` waves with
 * lds_bytes of LDS, law_words of them per body for a force law; false when
 * it does not fit. */
B3D_FN bool quad_layout(const Geometry& g, int waves, size_t lds_bytes, int law_words, QuadLayout* q) {
    if (g.max_s > 64 || g.max_b > 255 || g.max_c > 1023 || g.max_j > 16) return false;
    q->waves = waves;
    int hw = hit_words(g);
    q->hits = 4 * kShapeRows * g.max_s;
    q->jkeys = q->hits + hw + 1;
    int xa = q->jkeys + g.max_j;
    q->last = 0;
    q->pos = q->last + g.max_b;
    q->level = q->pos + g.max_c + 2;
    q->order = q->level + g.max_c;
    q->jlast = q->order + g.max_c;
    q->jlev = q->jlast + g.max_b;
    q->jgeo = q->jlev + g.max_j;
    q->jconst = q->jgeo + kJGWords * g.max_j;
    int xb = q->jconst + kJCWords * g.max_j;
    q->heads = xa > xb ? xa : xb;
    q->y = q->heads + g.max_c;
    q->bounds = q->y;
    q->masks = q->bounds + 6 * g.max_s;
    q->keys = q->masks + 2 * g.max_s;
    q->clip = q->keys + g.max_c;
    int most = (int)(lds_bytes / 4 - kQuadWgWords) / kQuadCols - law_words * g.max_b, room = most - q->clip;
    int rows = q->y + quad_body_rows(g);
    int cand = g.max_s * (g.max_s - 1) / 2;
    q->cw = room / kClipWords;
    if (q->cw > 4 * waves) q->cw = 4 * waves;
    if (q->cw > cand) q->cw = cand < 1 ? 1 : cand;
    if (q->cw < 4 && q->cw < cand) return false;
    int gen = q->clip + q->cw * kClipWords;
    q->law = gen > rows ? gen : rows;
    q->words = q->law + law_words * g.max_b;
    q->scratch_tile_words = (size_t)g.scr_words * kLanes + (size_t)kLanes * g.max_c * kQRecWords;
    return q->law <= most;
}

}  // namespace b3d

#endif
