/*
 * b3d_quad.h - one world's step on four lanes of each of a workgroup's
 * waves, for batches that leave most of the chip idle at one lane a world.
 *
 * A workgroup of W (8 or 4) waves steps kQuadCols = 16 worlds, a quarter of
 * a 64-world tile: lanes 4c .. 4c + 3 of every wave belong to world c, so a
 * world has 4 W lanes ("workers").  Two ways of using them:
 *   - what is independent within a world (shapes, candidate pairs, contact
 *     preparation, body updates, joint geometry) goes one item to a worker,
 *     through the same scalar functions as the other steps (b3d_lane.h with
 *     LDS rows of B3D_ROW = 16 words and the per-step records in LDS);
 *   - what is a chain (the Gauss-Seidel solves, whose order is part of the
 *     result) goes one solve to a quad of lanes: lane 0..2 of the quad holds
 *     component x, y, z of every vector, lane 3 the scalars that ride along,
 *     and products across components use DPP operands.
 * Why: a chain's time is its instruction count (a dependent fp32 operation
 * issues every ~5 cycles, whatever the other lanes or a second wave of the
 * SIMD do), and a vector operation on a quad is one instruction where one
 * lane needs three (a dot product 4 for 5, a cross product 5 for 9, a
 * matrix-vector product 5 for 15).  Every component is computed by the same
 * operations in the same order as in the scalar code, so the bits are the
 * same.
 *
 * Each wave owns contacts and joints for the whole step: joint j is wave
 * j mod W's, contact number i in level order wave i mod W's, and the owner keeps its rows in registers over all sweeps
 * (the first CR contacts and JR joints of a wave; further contacts are
 * loaded from their records for each solve).  The velocities are in LDS;
 * levels of contacts and of joint solves on disjoint dynamic bodies
 * (b3d_lane.h) go in turn with a workgroup barrier after each, which costs
 * ~50 cycles.
 *
 * Device only.  Include before any other header of the engine.
 */
#ifndef PUFFYSICS_AMD_B3D_QUAD_H
#define PUFFYSICS_AMD_B3D_QUAD_H

#include "b3d_quad_layout.h"

namespace b3d {

#define B3Q_FN static __device__ inline __attribute__((always_inline))

/* ---- quads: component arithmetic on DPP operands ---- */
template <int P>
B3Q_FN float qperm(float x) {
    return __builtin_bit_cast(float,
        __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), P, 0xf, 0xf, true));
}
/* lane P's value in all four lanes */
template <int P>
B3Q_FN float qbc(float x) { return qperm<P * 0x55>(x); }
B3Q_FN float qnext(float x) { return qperm<1 | 2 << 2 | 0 << 4 | 3 << 6>(x); }   /* y z x */
B3Q_FN float qprev(float x) { return qperm<2 | 0 << 2 | 1 << 4 | 3 << 6>(x); }   /* z x y */
B3Q_FN float qdot3(float a, float b) {
    float t = a * b;
    return qbc<0>(t) + qbc<1>(t) + qbc<2>(t);
}
B3Q_FN float qcross(float a, float b) { return qnext(a) * qprev(b) - qprev(a) * qnext(b); }
/* a lane's row of a matrix: its component of the three columns */
struct QM { float x, y, z; };
B3Q_FN float qmv(QM m, float v) { return m.x * qbc<0>(v) + m.y * qbc<1>(v) + m.z * qbc<2>(v); }
/* rot (03_math.inl) by the unit quaternion q (lane 3: s) */
B3Q_FN float qrot(float q, float v) {
    float t = qcross(q, v) * 2.0f;
    return v + (t * qbc<3>(q) + qcross(q, t));
}

/* One lane's view: its world (L, rows in LDS), its place in the quad and
 * among the world's workers. */
struct QLane {
    Lane L;
    float* lds;        /* LDS rows + world column */
    uint32_t* recs;    /* the world's contact records */
    PairStage st;      /* the tile's manifold stage */
    int sub, wave, worker;
    int waves, workers;   /* compile-time constants once inlined */
    QuadLayout q;
};
B3Q_FN float* lrow(const QLane& Q, int word) { return Q.lds + word * kRow; }
B3Q_FN int lgeti(const QLane& Q, int word) { return __builtin_bit_cast(int, Q.lds[word * kRow]); }
B3Q_FN void lseti(const QLane& Q, int word, int v) { Q.lds[word * kRow] = __builtin_bit_cast(float, v); }

/* ---- contact generation ---- */

/* The old contacts' keys, their pairs' order and warm data, the shape
 * records and bounds, and the joint keys (find_contacts' opening): one item
 * to a worker. */
B3Q_FN void quad_open(const QLane& Q, int old_n, int ns, int nj) {
    const Lane& L = Q.L;
    for (int k = Q.worker; k < old_n; k += Q.workers) {
        int sa = ldi(L.w, cw(L, k, C_SHAPE_A)), sb = ldi(L.w, cw(L, k, C_SHAPE_B));
        int pk = k > 0 ? k - 1 : 0;
        int pa = ldi(L.w, cw(L, pk, C_SHAPE_A)), pb = ldi(L.w, cw(L, pk, C_SHAPE_B));
        uint32_t key = shape_key(sa, sb);
        lseti(Q, Q.q.keys + k, (int)key);
        uint32_t* o = old_rec(L, k);
        sti(o, O_SHAPE_A, sa);
        sti(o, O_SHAPE_B, sb);
        if (k > 0 && !(shape_key(pa, pb) < key && (uint32_t)sa < 65536u && (uint32_t)sb < 65536u))
            lseti(Q, Q.q.hits + hit_words(L.g), 1);
    }
    old_warm_copy(L, old_n, Q.worker, Q.workers);
    shape_pass(L, ns, lrow(Q, Q.q.bounds), Q.worker, Q.workers);
    for (int j = Q.worker; j < nj; j += Q.workers) {
        uint32_t key = 0xffffffffu;
        if (!ldi(L.w, jw(L, j, J_COLLIDE_CONNECTED)))
            key = pair_key(ldi(L.w, jw(L, j, J_BODY_A)), ldi(L.w, jw(L, j, J_BODY_B)));
        lseti(Q, Q.q.jkeys + j, (int)key);
    }
}

B3Q_FN uint64_t quad_mask(const QLane& Q, int i) {
    return (uint64_t)(uint32_t)lgeti(Q, Q.q.masks + 2 * i) | ((uint64_t)(uint32_t)lgeti(Q, Q.q.masks + 2 * i + 1) << 32);
}
/* Bound-overlap masks, a row of pairs (i, j > i) to a worker. */
B3Q_FN void quad_overlaps(const QLane& Q, int ns) {
    const float* bounds = lrow(Q, Q.q.bounds);
    for (int i = Q.worker; i < ns; i += Q.workers) {
        Box6 bi = box_load(bounds + i * 6 * kRow);
        uint64_t m = 0;
        for (int j0 = i + 1; j0 < ns; j0 += 4) {
            Box6 bj[4];
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (j0 + k < ns) bj[k] = box_load(bounds + (j0 + k) * 6 * kRow);
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (j0 + k < ns && box_overlap(bi, bj[k])) m |= 1ull << (j0 + k);
        }
        lseti(Q, Q.q.masks + 2 * i, (int)(uint32_t)m);
        lseti(Q, Q.q.masks + 2 * i + 1, (int)(uint32_t)(m >> 32));
    }
}

/* This worker's share of the narrowphase: candidates worker, worker + cw,
 * ... in (i, j) order, their manifolds to the stage (pair_share).  The pair
 * is looked up first and collided outside that loop: the workers' pairs are
 * in different rows of the masks, and a collision inside the walk would run
 * once per row. */
B3Q_FN void quad_collide(const QLane& Q, int ns, int nj, int old_n) {
    const Lane& L = Q.L;
    if (Q.worker >= Q.q.cw) return;
    bool sorted = lgeti(Q, Q.q.hits + hit_words(L.g)) == 0;
    int acc = 0, i = 0;
    uint64_t m = ns > 0 ? quad_mask(Q, 0) : 0;
    float* clip = lrow(Q, Q.q.clip + Q.worker * kClipWords);
    for (int t = Q.worker;; t += Q.q.cw) {
        int c = __builtin_popcountll(m);
        while (i < ns && t >= acc + c) {
            acc += c;
            i++;
            m = i < ns ? quad_mask(Q, i) : 0;
            c = __builtin_popcountll(m);
        }
        if (i >= ns) break;
        uint64_t mm = m;
        for (int k = t - acc; k > 0; k--) mm &= mm - 1;
        int j = __builtin_ctzll(mm);
        PairShape A, B;
        pshape_load(L, i, &A);
        pshape_load(L, j, &B);
        uint32_t bkey = pair_key(A.body, B.body);
        int joined = 0;
        for (int k = 0; k < nj; k++) joined |= (uint32_t)lgeti(Q, Q.q.jkeys + k) == bkey;
        Mani mf;
        mf.count = 0;
        if (!(A.body == B.body || (A.bflags & B.bflags & kBodyStatic) || (A.cat & B.mask) == 0
                || (B.cat & A.mask) == 0 || joined))
            collide_pair(&mf, A.P, B.P, clip);
        if (mf.count > 0) {
            /* the old contact of the same pair (the merge of the sorted lists) */
            uint32_t key = shape_key(i, j);
            int match = -1;
            if (sorted) {
                int lo = 0, hi = old_n;
                while (lo < hi) {
                    int mid = (lo + hi) >> 1;
                    if ((uint32_t)lgeti(Q, Q.q.keys + mid) < key) lo = mid + 1;
                    else hi = mid;
                }
                if (lo < old_n && (uint32_t)lgeti(Q, Q.q.keys + lo) == key) match = lo;
            }
            mani_store(Q.st, L.lane, t, mf, key, match);
            lds_or(lrow(Q, Q.q.hits + (t >> 5)), 1u << (t & 31));
        }
    }
}

B3Q_FN Quad quad_of(V3 v, float s) {
    return Quad{__builtin_bit_cast(uint32_t, v.x), __builtin_bit_cast(uint32_t, v.y),
        __builtin_bit_cast(uint32_t, v.z), __builtin_bit_cast(uint32_t, s)};
}
B3Q_FN uint32_t* qrec(const QLane& Q, int c) { return Q.recs + (size_t)c * kQRecWords; }

/* New contact k of the world: the candidate with the k-th manifold, written
 * to the world's row (write_new_contact) and prepared (contact_prep,
 * b3_prepare_one_contact) into its record, with its head in LDS.  Returns
 * its CF_* flags. */
B3Q_FN int quad_contact(const QLane& Q, int k, int t, int old_n, bool sorted, Soft cs, Soft ss) {
    const Lane& L = Q.L;
    uint32_t* w = L.w;
    Mani m;
    uint32_t key;
    int match;
    mani_load(Q.st, L.lane, t, &m, &key, &match);
    int i = (int)(key >> 16), j = (int)(key & 0xffffu);
    PairShape A, B;
    pshape_load(L, i, &A);
    pshape_load(L, j, &B);
    OldWarm orec;
    if (sorted && match >= 0) old_load(L, match, &orec);
    /* zero unless the body is dynamic (08:236-241) */
    float ma = 0.0f, mb = 0.0f;
    M3 ia = m3zero(), ib = m3zero();
    if (A.bflags & kBodyDynamic) {
        ma = ldf(w, bw(L, A.body, B_INV_MASS));
        ia = ldm3(w, bw(L, A.body, B_INV_I_WORLD));
    }
    if (B.bflags & kBodyDynamic) {
        mb = ldf(w, bw(L, B.body, B_INV_MASS));
        ib = ldm3(w, bw(L, B.body, B_INV_I_WORLD));
    }
    uint32_t flags_a = ldu(w, bw(L, A.body, B_FLAGS)), flags_b = ldu(w, bw(L, B.body, B_FLAGS));
    NewContact nc = new_contact(L, i, j, A, B, m, sorted, match, orec, old_n);
    int info = store_new_contact(L, k, i, j, A, B, nc);
    const int keep = (L.opts & kKeepSolverFields) != 0;
    const int need_rv = keep || (info & CF_RESTITUTION);
    V3 va = zero3(), wa = zero3(), vb = zero3(), wb = zero3();
    if (need_rv) {
        /* the bodies' velocities of the start of the step */
        va = ld3(w, bw(L, A.body, B_LIN_VEL));
        wa = ld3(w, bw(L, A.body, B_ANG_VEL));
        vb = ld3(w, bw(L, B.body, B_LIN_VEL));
        wb = ld3(w, bw(L, B.body, B_ANG_VEL));
    }
    ContactPrep p = contact_prep(nc.count, nc.normal, nc.t1, nc.r_a, nc.r_b, nc.base_sep, nc.ni, ma, mb, ia, ib,
        need_rv, va, wa, vb, wb);
    if (keep) keep_solver_fields(L, k, nc.count, p, ma, mb, ia, ib, (info & CF_STATIC) ? ss : cs);
    Quad* r = reinterpret_cast<Quad*>(qrec(Q, k));
    float friction = sqrtf(A.friction * B.friction);
    float restitution = A.restitution > B.restitution ? A.restitution : B.restitution;
    float rolling = maxf(A.rolling, B.rolling);
    r[QR_N] = quad_of(nc.normal, friction);
    r[QR_T1] = quad_of(nc.t1, p.twist_mass);
    r[QR_CA] = quad_of(p.center_a, rolling);
    r[QR_CB] = quad_of(p.center_b, restitution);
    r[QR_IA] = quad_of(ia.cx, ma);
    r[QR_IA + 1] = quad_of(ia.cy, p.tmass.cx.x);
    r[QR_IA + 2] = quad_of(ia.cz, p.tmass.cx.y);
    r[QR_IB] = quad_of(ib.cx, mb);
    r[QR_IB + 1] = quad_of(ib.cy, p.tmass.cy.y);
    r[QR_IB + 2] = quad_of(ib.cz, 0.0f);
    r[QR_ROLL] = quad_of(nc.roll, nc.twist);
    r[QR_FI] = quad_of(v3(nc.fi.x, nc.fi.y, 0.0f), 0.0f);
    r[QR_NMASS] = quad_of(v3(p.nmass[0], p.nmass[1], p.nmass[2]), p.nmass[3]);
    r[QR_NI] = quad_of(v3(p.ni[0], p.ni[1], p.ni[2]), p.ni[3]);
    r[QR_TN] = quad_of(zero3(), 0.0f);
    r[QR_LEVER] = quad_of(v3(p.lever[0], p.lever[1], p.lever[2]), p.lever[3]);
    r[QR_SEP] = quad_of(v3(p.base_sep[0], p.base_sep[1], p.base_sep[2]), p.base_sep[3]);
    r[QR_RV] = quad_of(v3(p.rel_vel[0], p.rel_vel[1], p.rel_vel[2]), p.rel_vel[3]);
#pragma unroll
    for (int q = 0; q < kMaxManifold; q++) {
        if (q >= nc.count) continue;
        r[QR_RA + q] = quad_of(nc.r_a[q], 0.0f);
        r[QR_RB + q] = quad_of(nc.r_b[q], 0.0f);
    }
    /* the head's CF_DYN_* are the bodies' flags, which decide what a solve
     * writes, whatever their type (read here, by all workers, rather than in
     * quad_levels: at 4,096 worlds the arm 144.1 -> 143.3 us, the bin 397 ->
     * 392) */
    int levels = (info & ~(CF_DYN_A | CF_DYN_B)) | (flags_a & kFlagDynamic ? CF_DYN_A : 0)
        | (flags_b & kFlagDynamic ? CF_DYN_B : 0);
    lseti(Q, Q.q.heads + k, A.body | (B.body << 8) | (nc.count << 16) | (levels << 20));
    return info;
}

/* The world's new contacts, one to a worker at a time, and its header
 * counts (append_share, find_pairs).  Returns the contact count. */
B3Q_FN int quad_append(const QLane& Q, int old_n, Soft cs, Soft ss, int* wg) {
    const Lane& L = Q.L;
    int total = 0, hw = hit_words(L.g);
    for (int k = 0; k < hw; k++) total += __builtin_popcount((uint32_t)lgeti(Q, Q.q.hits + k));
    int cc = total < L.g.max_c ? total : L.g.max_c;
    bool sorted = lgeti(Q, Q.q.hits + hw) == 0;
    int acc = 0, word = 0, flags = 0;
    for (int k = Q.worker; k < cc; k += Q.workers) {
        uint32_t bits = (uint32_t)lgeti(Q, Q.q.hits + word);
        while (acc + __builtin_popcount(bits) <= k) {
            acc += __builtin_popcount(bits);
            word++;
            bits = (uint32_t)lgeti(Q, Q.q.hits + word);
        }
        for (int r = k - acc; r > 0; r--) bits &= bits - 1;
        flags |= quad_contact(Q, k, word * 32 + __builtin_ctz(bits), old_n, sorted, cs, ss);
    }
    if (flags & CF_RESTITUTION) atomicOr(wg + WG_REST, 1);
    if (Q.worker == 0) {
        sti(L.w, H_CONTACT_COUNT, cc);
        sti(L.w, H_CONTACT_OVERFLOW, ldi(L.w, H_CONTACT_OVERFLOW) | (total > L.g.max_c ? 1 : 0));
        sti(L.w, H_CONTACTS_DROPPED, ldi(L.w, H_CONTACTS_DROPPED) + (total - cc));
    }
    return cc;
}

/* The contacts' levels (sched_build) and their order by level: entry i is
 * contact | level << 10.  One worker of the world. */
B3Q_FN void quad_levels(const QLane& Q, int cc, int nb, int* wg) {
    for (int b = 0; b < nb; b++) lseti(Q, Q.q.last + b, 0);
    for (int lev = 0; lev <= cc; lev++) lseti(Q, Q.q.pos + lev, 0);
    int nlev = 0;
    for (int c0 = 0; c0 < cc; c0 += kSchedChunk) {
        int hd[kSchedChunk];
#pragma unroll
        for (int k = 0; k < kSchedChunk; k++)
            if (c0 + k < cc) hd[k] = lgeti(Q, Q.q.heads + c0 + k);
#pragma unroll
        for (int k = 0; k < kSchedChunk; k++) {
            int c = c0 + k;
            if (c >= cc) continue;
            int a = hd[k] & 255, b = (hd[k] >> 8) & 255, fl = hd[k] >> 20;
            int la = (fl & CF_DYN_A) ? lgeti(Q, Q.q.last + a) : 0;
            int lb = (fl & CF_DYN_B) ? lgeti(Q, Q.q.last + b) : 0;
            int lev = (la > lb ? la : lb) + 1;
            if (fl & CF_DYN_A) lseti(Q, Q.q.last + a, lev);
            if (fl & CF_DYN_B) lseti(Q, Q.q.last + b, lev);
            lseti(Q, Q.q.level + c, lev);
            lseti(Q, Q.q.pos + lev, lgeti(Q, Q.q.pos + lev) + 1);
            if (lev > nlev) nlev = lev;
        }
    }
    int run = 0;
    for (int lev = 1; lev <= nlev; lev++) {
        int n = lgeti(Q, Q.q.pos + lev);
        lseti(Q, Q.q.pos + lev, run);
        run += n;
    }
    for (int c = 0; c < cc; c++) {
        int lev = lgeti(Q, Q.q.level + c);
        int at = lgeti(Q, Q.q.pos + lev);
        lseti(Q, Q.q.pos + lev, at + 1);
        lseti(Q, Q.q.order + at, c | (lev << 10));
    }
    atomicMax(wg + WG_LEVELS, nlev);
}

/* The joint solves' levels (joint_levels_scan): of joint j in the pass's
 * two iterations, at jlev + j (first | second << 8).  One worker. */
B3Q_FN void quad_joint_levels(const QLane& Q, int nj, int nb, int* wg) {
    const Lane& L = Q.L;
    for (int b = 0; b < nb; b++) lseti(Q, Q.q.jlast + b, 0);
    int nlev = 0;
    for (int it = 0; it < kJointIters; it++) {
        for (int j = 0; j < nj; j++) {
            uint32_t ab = ldu(joint_rec(L, j), JS_AB);
            int a = (int)(ab & 0xffffu), b = (int)(ab >> 16);
            bool da = is_dyn_flag(L, a), db = is_dyn_flag(L, b);
            int la = da ? lgeti(Q, Q.q.jlast + a) : 0;
            int lb = db ? lgeti(Q, Q.q.jlast + b) : 0;
            int lev = (la > lb ? la : lb) + 1;
            /* no dynamic body keeps the two solves of its row apart */
            if (!da && !db) lev = 1 + it;
            if (da) lseti(Q, Q.q.jlast + a, lev);
            if (db) lseti(Q, Q.q.jlast + b, lev);
            lseti(Q, Q.q.jlev + j, it == 0 ? lev : lgeti(Q, Q.q.jlev + j) | (lev << 8));
            if (lev > nlev) nlev = lev;
        }
    }
    atomicMax(wg + WG_JLEVELS, nlev);
    atomicMax(wg + WG_JOINTS, nj);
}

B3Q_FN M3 rm3(const uint32_t* r, int k) { M3 m; m.cx = r3(r, k); m.cy = r3(r, k + 3); m.cz = r3(r, k + 6); return m; }
/* A joint's constants (JC_*), as prepare_joints left them in the world and
 * the joint record. */
struct JConst { uint32_t ab; int info; b3d::Q qa, qb; V3 pa, pb, dc; float ma, mb; M3 ia, ib; };
B3Q_FN JConst jconst_world(const Lane& L, int j) {
    const uint32_t* w = L.w;
    return JConst{ldu(joint_rec(L, j), JS_AB), ldi(joint_rec(L, j), JS_INFO), ldq(w, jw(L, j, J_FRAME_Q_A)),
        ldq(w, jw(L, j, J_FRAME_Q_B)), ld3(w, jw(L, j, J_FRAME_P_A)), ld3(w, jw(L, j, J_FRAME_P_B)),
        ld3(w, jw(L, j, J_DELTA_CENTER)), ldf(w, jw(L, j, J_INV_MASS_A)), ldf(w, jw(L, j, J_INV_MASS_B)),
        ldm3(w, jw(L, j, J_INV_I_A)), ldm3(w, jw(L, j, J_INV_I_B))};
}
B3Q_FN void jconst_store(uint32_t* c, const JConst& k) {
    rsu(c, JC_AB, k.ab);
    rsu(c, JC_INFO, (uint32_t)k.info);
    rsq(c, JC_QA, k.qa);
    rsq(c, JC_QB, k.qb);
    rs3(c, JC_PA, k.pa);
    rs3(c, JC_PB, k.pb);
    rs3(c, JC_DC, k.dc);
    rsf(c, JC_MA, k.ma);
    rsf(c, JC_MB, k.mb);
    rs3(c, JC_IA, k.ia.cx);
    rs3(c, JC_IA + 3, k.ia.cy);
    rs3(c, JC_IA + 6, k.ia.cz);
    rs3(c, JC_IB, k.ib.cx);
    rs3(c, JC_IB + 3, k.ib.cy);
    rs3(c, JC_IB + 6, k.ib.cz);
}
B3Q_FN JConst jconst_load(const uint32_t* c) {
    return JConst{ru(c, JC_AB), (int)ru(c, JC_INFO), rq4(c, JC_QA), rq4(c, JC_QB), r3(c, JC_PA), r3(c, JC_PB),
        r3(c, JC_DC), rf(c, JC_MA), rf(c, JC_MB), rm3(c, JC_IA), rm3(c, JC_IB)};
}

/* The joints' delta-pose geometry (joint_geo) to their LDS rows.  The
 * waves take one of three parts each, so that no lane runs all of it: waves
 * 0, 3, .. the anchors, separation and twist (a weld: the angular error),
 * 1, 4, .. the point rows' inverse matrix, 2, 5, .. the hinge rows and their
 * matrix.  Waves `first` and up take part.  The first call of a step reads
 * the constants from memory and leaves them in LDS for the others (from
 * memory each time, eight hinges' geometry took 2.6 us a substep). */
template <bool First>
B3Q_FN void quad_joint_geometry(const QLane& Q, int nj, int first) {
    const Lane& L = Q.L;
    int wv = Q.wave - first, n = Q.waves - first;
    if (wv < 0) return;
    int parts = n < 3 ? n : 3, part = wv % parts;
    int stride = 4 * ((n - part + parts - 1) / parts);
    for (int j = (wv / parts) * 4 + Q.sub; j < nj; j += stride) {
        uint32_t* crow = (uint32_t*)lrow(Q, Q.q.jconst + j * kJCWords);
        JConst c = First ? jconst_world(L, j) : jconst_load(crow);
        if (First && part == 0) jconst_store(crow, c);
        const int info = c.info;
        const b3d::Q fqa = c.qa, fqb = c.qb;
        const V3 fpa = c.pa, fpb = c.pb, dcen = c.dc;
        const float ma = c.ma, mb = c.mb;
        const M3 ia = c.ia, ib = c.ib;
        const uint32_t* da = delta_rec(L, (int)(c.ab & 0xffffu));
        const uint32_t* db = delta_rec(L, (int)(c.ab >> 16));
        b3d::Q dqa = rq4(da, BD_DQ), dqb = rq4(db, BD_DQ);
        V3 dpa = r3(da, BD_DP), dpb = r3(db, BD_DP);
        float* g = lrow(Q, Q.q.jgeo + j * kJGWords);
        auto put = [g](int quad, int k, float v) { g[(4 * quad + k) * kRow] = v; };
        auto put3 = [put](int quad, V3 v) { put(quad, 0, v.x); put(quad, 1, v.y); put(quad, 2, v.z); };
        /* the unused results of each part's call fall away */
        bool fixed = (info & JF_FIXED) != 0, weld = (info & JF_WELD) != 0;
        if (part == 0 || parts < 2) {
            JGeo o = joint_geo(info, dqa, dqb, dpa, dpb, fqa, fqb, fpa, fpb, dcen, ma, mb, ia, ib);
            put3(JG_RA_TW, o.ra);
            put3(JG_RB_RELX, o.rb);
            put3(JG_PSEP_RELY, o.psep);
            if (weld) {
                if (!fixed) put3(JG_PY_KXY, o.cv);
            } else {
                put(JG_RA_TW, 3, o.tw);
                put(JG_RB_RELX, 3, o.relx);
                put(JG_PSEP_RELY, 3, o.rely);
            }
        }
        if (part == 1 || parts < 2) {
            M3 pki = inv3(point_k(ma, mb, ia, ib, rot(dqa, fpa), rot(dqb, fpb)));
            put3(JG_K0_KYY, pki.cx);
            put3(JG_K1_KINV, pki.cy);
            put3(JG_K2, pki.cz);
        }
        if ((part == 2 || parts < 3) && part == parts - 1 && !weld && !fixed) {
            JGeo o = joint_geo(info & ~(JF_SPRING | JF_MOTOR | JF_LIMIT), dqa, dqb, dpa, dpb, fqa, fqb, fpa, fpb, dcen,
                ma, mb, ia, ib);
            put3(JG_PX_KXX, o.px);
            put3(JG_PY_KXY, o.py);
            put(JG_PX_KXX, 3, o.kxx);
            put(JG_PY_KXY, 3, o.kxy);
            put(JG_K0_KYY, 3, o.kyy);
            put(JG_K1_KINV, 3, o.kinv);
        }
    }
}

/* ---- contact rows on quads ---- */

/* A contact's row in a quad's registers: each float is one quad of the
 * record, lane 3 holding the scalar that rides along (QR_*): friction with
 * n, twist mass with t1, rolling with ca, restitution with cb, the inverse
 * masses and the tangent mass with the inertia columns, the twist impulse
 * with roll.  Of the per-point values (nmass, ni, tn, lever, sep) lane p
 * holds point p's. */
struct CQ {
    int c, lev, fl;        /* contact (-1: none), its level, CF_* flags | points << 8; the bodies' velocity rows */
    int va, vb;
    float n, t1, ca, cb, roll, fi, nmass, ni, tn, lever, sep;
    QM ia, ib;
    float ra[kMaxManifold], rb[kMaxManifold];
};
constexpr int kQDynA = 1 << 16, kQDynB = 1 << 17;   /* CQ::fl, JQ::info: the body's velocity is written */

B3Q_FN float qload(const uint32_t* r, int quad) { return __builtin_bit_cast(float, r[4 * quad]); }
/* Velocity rows: this lane's component (lane 3: a pad word). */
B3Q_FN int qvel_row(int b) { return b * kVelWords * kRow; }
B3Q_FN float* qvel(const QLane& Q) { return Q.L.vel + Q.sub * kRow; }

/* This lane's part of the row of order entry e (contact | level << 10),
 * with its separations at the bodies' delta poses (08_contacts.inl:
 * 331-333). */
B3Q_FN void cq_deltas(const QLane& Q, const CQ& r, float* dpa, float* dqa, float* dpb, float* dqb) {
    int d = Q.q.y + quad_delta_word(Q.L.g) + Q.sub;
    int a = r.va / (kVelWords * kRow), b = r.vb / (kVelWords * kRow);
    const float* da = lrow(Q, d + a * 4 * kDeltaRows);
    const float* db = lrow(Q, d + b * 4 * kDeltaRows);
    *dpa = da[BD_DP * kRow];
    *dqa = da[BD_DQ * kRow];
    *dpb = db[BD_DP * kRow];
    *dqb = db[BD_DQ * kRow];
}
B3Q_FN float cq_separations(const QLane& Q, const CQ& r, float base) {
    float dpa, dqa, dpb, dqb;
    cq_deltas(Q, r, &dpa, &dqa, &dpb, &dqb);
    float dp = dpb - dpa, sep = 0.0f;
#pragma unroll
    for (int p = 0; p < kMaxManifold; p++) {
        if (p >= ((r.fl >> 8) & 255)) continue;
        float ds = dp + (qrot(dqb, r.rb[p]) - qrot(dqa, r.ra[p]));
        float s = qdot3(ds, r.n);
        sep = Q.sub == p ? s : sep;
    }
    return sep + base;
}
B3Q_FN void cq_load(const QLane& Q, int e, CQ* r) {
    int c = e & 1023;
    int hd = lgeti(Q, Q.q.heads + c);
    const uint32_t* rc = qrec(Q, c) + Q.sub;
    int a = hd & 255, b = (hd >> 8) & 255;
    r->c = c;
    r->lev = e >> 10;
    r->fl = (hd >> 20) | (((hd >> 16) & 15) << 8) | (is_dyn_flag(Q.L, a) ? kQDynA : 0)
        | (is_dyn_flag(Q.L, b) ? kQDynB : 0);
    r->va = qvel_row(a);
    r->vb = qvel_row(b);
    r->n = qload(rc, QR_N);
    r->t1 = qload(rc, QR_T1);
    r->ca = qload(rc, QR_CA);
    r->cb = qload(rc, QR_CB);
    r->roll = qload(rc, QR_ROLL);
    r->fi = qload(rc, QR_FI);
    r->nmass = qload(rc, QR_NMASS);
    r->ni = qload(rc, QR_NI);
    r->tn = qload(rc, QR_TN);
    r->lever = qload(rc, QR_LEVER);
    r->ia = QM{qload(rc, QR_IA), qload(rc, QR_IA + 1), qload(rc, QR_IA + 2)};
    r->ib = QM{qload(rc, QR_IB), qload(rc, QR_IB + 1), qload(rc, QR_IB + 2)};
#pragma unroll
    for (int p = 0; p < kMaxManifold; p++) {
        r->ra[p] = 0.0f;
        r->rb[p] = 0.0f;
        if (p >= ((r->fl >> 8) & 255)) continue;
        r->ra[p] = qload(rc, QR_RA + p);
        r->rb[p] = qload(rc, QR_RB + p);
    }
}
/* The base separations a row's separations add (kept in the record). */
B3Q_FN float cq_base(const QLane& Q, const CQ& r) { return qload(qrec(Q, r.c) + Q.sub, QR_SEP); }
/* The row's impulses back to the record. */
B3Q_FN void cq_store(const QLane& Q, const CQ& r) {
    uint32_t* rc = qrec(Q, r.c) + Q.sub;
    rc[4 * QR_NI] = __builtin_bit_cast(uint32_t, r.ni);
    rc[4 * QR_TN] = __builtin_bit_cast(uint32_t, r.tn);
    rc[4 * QR_FI] = __builtin_bit_cast(uint32_t, r.fi);
    rc[4 * QR_ROLL] = __builtin_bit_cast(uint32_t, r.roll);
}

/* A row's bodies' velocities: read, and written back where dynamic. */
struct QVel { float va, wa, vb, wb; };
B3Q_FN QVel qvel_load(const QLane& Q, int va, int vb) {
    const float* v = qvel(Q);
    return QVel{v[va], v[va + kVelAng * kRow], v[vb], v[vb + kVelAng * kRow]};
}
B3Q_FN void qvel_store(const QLane& Q, int va, int vb, int fl, QVel x) {
    float* v = qvel(Q);
    if (fl & kQDynA) {
        v[va] = x.va;
        v[va + kVelAng * kRow] = x.wa;
    }
    if (fl & kQDynB) {
        v[vb] = x.vb;
        v[vb + kVelAng * kRow] = x.wb;
    }
}
/* Impulse P at levers ra and rb on the bodies (b after a, opposite). */
B3Q_FN void qimpulse(QVel* x, float ma, QM ia, float mb, QM ib, float ra, float rb, float P) {
    x->va = x->va - ma * P;
    x->wa = x->wa - qmv(ia, qcross(ra, P));
    x->vb = x->vb + mb * P;
    x->wb = x->wb + qmv(ib, qcross(rb, P));
}

/* The contact's warm start (08:194-232). */
B3Q_FN void cq_warm(const QLane& Q, const CQ& r) {
    QVel x = qvel_load(Q, r.va, r.vb);
    float ma = qbc<3>(r.ia.x), mb = qbc<3>(r.ib.x);
#pragma unroll
    for (int p = 0; p < kMaxManifold; p++) {
        if (p >= ((r.fl >> 8) & 255)) continue;
        float ni = p == 0 ? qbc<0>(r.ni) : (p == 1 ? qbc<1>(r.ni) : (p == 2 ? qbc<2>(r.ni) : qbc<3>(r.ni)));
        qimpulse(&x, ma, r.ia, mb, r.ib, r.ra[p], r.rb[p], r.n * ni);
    }
    float t2 = qcross(r.t1, r.n);
    float f = r.t1 * qbc<0>(r.fi) + t2 * qbc<1>(r.fi);
    qimpulse(&x, ma, r.ia, mb, r.ib, r.ca, r.cb, f);
    float tr = r.n * qbc<3>(r.roll) + r.roll;
    x.wa = x.wa - qmv(r.ia, tr);
    x.wb = x.wb + qmv(r.ib, tr);
    qvel_store(Q, r.va, r.vb, r.fl, x);
}

/* Rolling resistance (07_packed.inl:24-45) on quads. */
B3Q_FN void cq_rolling(const CQ& r, float t2, float rolling, float total_n, float* impulse, QVel* x) {
    QM is = QM{r.ia.x + r.ib.x, r.ia.y + r.ib.y, r.ia.z + r.ib.z};
    M2 k;
    float it2 = qmv(is, t2);
    k.cx.x = qdot3(r.t1, qmv(is, r.t1));
    k.cy.y = qdot3(t2, it2);
    k.cx.y = qdot3(r.t1, it2);
    k.cy.x = k.cx.y;
    float wr = x->wb - x->wa;
    V2 rhs;
    rhs.x = qdot3(wr, r.t1);
    rhs.y = qdot3(wr, t2);
    V2 d = mv2(inv2(k), rhs);
    float next = *impulse - (r.t1 * d.x + t2 * d.y);
    float limit = rolling * total_n;
    float l2 = qdot3(next, next);
    if (l2 > limit * limit && l2 > 0.0f) next = next * rsqrt_scale(limit, l2);
    float delta = next - *impulse;
    *impulse = next;
    x->wa = x->wa - qmv(r.ia, delta);
    x->wb = x->wb + qmv(r.ib, delta);
}

/* One contact's solve, b3_solve_one_contact (08:315-413), as crow_solve. */
template <bool Relax>
B3Q_FN void cq_solve(const QLane& Q, CQ& r, float inv_h, float contact_speed, Soft cs, Soft ss) {
    QVel x = qvel_load(Q, r.va, r.vb);
    float ma = qbc<3>(r.ia.x), mb = qbc<3>(r.ib.x);
    /* each lane the coefficients of its own point */
    float vbias = 0.0f, mscale = 1.0f, iscale = 0.0f;
    if (!Relax) {
        bool st = (r.fl & CF_STATIC) != 0;
        float ms = st ? ss.mass_scale : cs.mass_scale;
        vbias = maxf(ms * (st ? ss.bias_rate : cs.bias_rate) * r.sep, -contact_speed);
        mscale = ms;
        iscale = st ? ss.impulse_scale : cs.impulse_scale;
    }
    if (r.sep > 0.0f) {
        vbias = r.sep * inv_h;
        mscale = 1.0f;
        iscale = 0.0f;
    }
#pragma unroll
    for (int p = 0; p < kMaxManifold; p++) {
        if (p >= ((r.fl >> 8) & 255)) continue;
        float vra = x.va + qcross(x.wa, r.ra[p]);
        float vrb = x.vb + qcross(x.wb, r.rb[p]);
        float vn = qdot3(vrb - vra, r.n);
        float dimp = -r.nmass * (mscale * vn + vbias) - iscale * r.ni;
        float nimp = maxf(r.ni + dimp, 0.0f);
        dimp = nimp - r.ni;
        r.ni = Q.sub == p ? nimp : r.ni;
        r.tn = Q.sub == p ? r.tn + nimp : r.tn;
        dimp = p == 0 ? qbc<0>(dimp) : (p == 1 ? qbc<1>(dimp) : (p == 2 ? qbc<2>(dimp) : qbc<3>(dimp)));
        qimpulse(&x, ma, r.ia, mb, r.ib, r.ra[p], r.rb[p], r.n * dimp);
    }
    if (Relax) {
        /* sums over the points, in point order */
        float lev = r.lever * r.ni;
        int pc = (r.fl >> 8) & 255;
        float total_n = 0.0f, twist_lim = 0.0f;
        if (pc > 0) {
            total_n = total_n + qbc<0>(r.ni);
            twist_lim = twist_lim + qbc<0>(lev);
        }
        if (pc > 1) {
            total_n = total_n + qbc<1>(r.ni);
            twist_lim = twist_lim + qbc<1>(lev);
        }
        if (pc > 2) {
            total_n = total_n + qbc<2>(r.ni);
            twist_lim = twist_lim + qbc<2>(lev);
        }
        if (pc > 3) {
            total_n = total_n + qbc<3>(r.ni);
            twist_lim = twist_lim + qbc<3>(lev);
        }
        float friction = qbc<3>(r.n), twist_imp = qbc<3>(r.roll);
        float twist_s = qdot3(r.n, x.wb - x.wa);
        float max_t = friction * twist_lim;
        float dtw = -qbc<3>(r.t1) * twist_s;
        float new_t = clampf(twist_imp + dtw, -max_t, max_t);
        dtw = new_t - twist_imp;
        float tw = r.n * dtw;
        x.wa = x.wa - qmv(r.ia, tw);
        x.wb = x.wb + qmv(r.ib, tw);

        float t2 = qcross(r.t1, r.n);
        float vr = (x.vb + qcross(x.wb, r.cb)) - (x.va + qcross(x.wa, r.ca));
        V2 vt;
        vt.x = qdot3(vr, r.t1);
        vt.y = qdot3(vr, t2);
        M2 tm;
        tm.cx.x = qbc<3>(r.ia.y);
        tm.cx.y = qbc<3>(r.ia.z);
        tm.cy.x = tm.cx.y;
        tm.cy.y = qbc<3>(r.ib.y);
        V2 tmv = mv2(tm, vt);
        float fx = qbc<0>(r.fi), fy = qbc<1>(r.fi);
        V2 ni;
        ni.x = fx - tmv.x;
        ni.y = fy - tmv.y;
        float max_f = friction * total_n;
        float fl2 = ni.x * ni.x + ni.y * ni.y;
        if (fl2 > max_f * max_f && fl2 > 0.0f) {
            float sc = rsqrt_scale(max_f, fl2);
            ni.x *= sc;
            ni.y *= sc;
        }
        r.fi = Q.sub == 0 ? ni.x : ni.y;
        float P = r.t1 * (ni.x - fx) + t2 * (ni.y - fy);
        qimpulse(&x, ma, r.ia, mb, r.ib, r.ca, r.cb, P);
        float roll = r.roll;
        if (r.fl & CF_ROLLING) cq_rolling(r, t2, qbc<3>(r.ca), total_n, &roll, &x);
        r.roll = Q.sub == 3 ? new_t : roll;
    }
    qvel_store(Q, r.va, r.vb, r.fl, x);
}

/* b3_apply_restitution for one contact (08:439-480). */
B3Q_FN void cq_restitution(const QLane& Q, CQ& r, float threshold) {
    if (!(r.fl & CF_RESTITUTION)) return;
    QVel x = qvel_load(Q, r.va, r.vb);
    float ma = qbc<3>(r.ia.x), mb = qbc<3>(r.ib.x), e = qbc<3>(r.cb);
    float rv = qload(qrec(Q, r.c) + Q.sub, QR_RV);
    /* each lane its own point's test: 1 when the point is left alone */
    float skip = rv > -threshold || r.tn == 0.0f ? 1.0f : 0.0f;
#pragma unroll
    for (int p = 0; p < kMaxManifold; p++) {
        if (p >= ((r.fl >> 8) & 255)) continue;
        float s = p == 0 ? qbc<0>(skip) : (p == 1 ? qbc<1>(skip) : (p == 2 ? qbc<2>(skip) : qbc<3>(skip)));
        if (s != 0.0f) continue;
        float vra = x.va + qcross(x.wa, r.ra[p]);
        float vrb = x.vb + qcross(x.wb, r.rb[p]);
        float vn = qdot3(vrb - vra, r.n);
        float imp = -r.nmass * (vn + e * rv);
        float nimp = maxf(r.ni + imp, 0.0f);
        imp = nimp - r.ni;
        r.ni = Q.sub == p ? nimp : r.ni;
        imp = p == 0 ? qbc<0>(imp) : (p == 1 ? qbc<1>(imp) : (p == 2 ? qbc<2>(imp) : qbc<3>(imp)));
        qimpulse(&x, ma, r.ia, mb, r.ib, r.ra[p], r.rb[p], r.n * imp);
    }
    qvel_store(Q, r.va, r.vb, r.fl, x);
}

/* The accumulated impulses of a row to the world's contact (contact_writeback). */
B3Q_FN void cq_writeback(const QLane& Q, const CQ& r) {
    const Lane& L = Q.L;
    uint32_t* w = L.w;
    if (Q.sub < ((r.fl >> 8) & 255)) {
        stf(w, pw(L, r.c, Q.sub, P_NORMAL_IMPULSE), r.ni);
        stf(w, pw(L, r.c, Q.sub, P_TOTAL_NORMAL), r.tn);
    }
    if (Q.sub < 2) stf(w, cw(L, r.c, C_FRICTION_IMPULSE + Q.sub), r.fi);
    if (Q.sub == 3) stf(w, cw(L, r.c, C_TWIST_IMPULSE), r.roll);
    else if (r.fl & CF_ROLLING) stf(w, cw(L, r.c, C_ROLLING_IMPULSE + Q.sub), r.roll);
}

/* ---- joint rows on quads ---- */

/* A joint's row in a quad's registers: vectors with a scalar of the row in
 * lane 3 (behind the slash), and two quads of scalars.
 *   ia, ib   inverse inertia columns / ma, lower, upper and mb, softness
 *            bias and mass scale
 *   axis, ia_ax, ib_ax, px, py, ra, rb, psep, pki  as JRow's / (geometry)
 *            twist, relx, rely with ra, rb, psep; kxx, kxy with px, py; kyy,
 *            kinv with pki
 *   s1       spring softness, then the softness' impulse scale
 *   s2       axial mass, torque limit, target, speed
 * A weld: axis its accumulated angular impulse, ia_ax, ib_ax, px its angular
 * mass columns / angular spring, py the angular error, s1 the linear spring,
 * s2 the linear and angular hertz. */
struct JQ {
    int j, lev, info;      /* joint (-1: none), its two levels (quad_joint_levels), JF_* | kQDyn* */
    int va, vb;
    QM ia, ib, pki;
    float lin_imp, ra, rb, psep, axis, ia_ax, ib_ax, px, py, s1, s2;
    float spring_imp, motor_imp, lower_imp, upper_imp, perp_x, perp_y;
};
/* The row's delta-pose geometry (quad_joint_geometry). */
B3Q_FN void jq_geometry(const QLane& Q, JQ* r) {
    const float* g = lrow(Q, Q.q.jgeo + r->j * kJGWords + Q.sub);
    auto v = [g](int quad) { return g[4 * quad * kRow]; };
    r->ra = v(JG_RA_TW);
    r->rb = v(JG_RB_RELX);
    r->psep = v(JG_PSEP_RELY);
    r->pki = QM{v(JG_K0_KYY), v(JG_K1_KINV), v(JG_K2)};
    r->py = v(JG_PY_KXY);
    if (!(r->info & JF_WELD)) r->px = v(JG_PX_KXX);
}
B3Q_FN void jq_load(const QLane& Q, int j, JQ* r) {
    const Lane& L = Q.L;
    const uint32_t* w = L.w;
    const uint32_t* rec = joint_rec(L, j);
    int k = Q.sub;
    bool l3 = k == 3;
    /* the vector at word f, word g in lane 3 */
    auto v = [w, k, l3, &L, j](int f, int g) { return ldf(w, jw(L, j, l3 ? g : f + k)); };
    auto s = [w, &L, j](int f) { return ldf(w, jw(L, j, f)); };
    auto pick = [k](int a, int b, int c, int d) { return k == 0 ? a : (k == 1 ? b : (k == 2 ? c : d)); };
    uint32_t ab = ldu(rec, JS_AB);
    int a = (int)(ab & 0xffffu), b = (int)(ab >> 16);
    r->j = j;
    r->lev = lgeti(Q, Q.q.jlev + j);
    r->info = ldi(rec, JS_INFO) | (is_dyn_flag(L, a) ? kQDynA : 0) | (is_dyn_flag(L, b) ? kQDynB : 0);
    r->va = qvel_row(a);
    r->vb = qvel_row(b);
    r->lin_imp = v(J_LINEAR_IMPULSE, J_LINEAR_IMPULSE);
    r->ia.x = v(J_INV_I_A, J_INV_MASS_A);
    r->ib.x = v(J_INV_I_B, J_INV_MASS_B);
    r->ia.y = v(J_INV_I_A + 3, J_LOWER_ANGLE);
    r->ia.z = v(J_INV_I_A + 6, J_UPPER_ANGLE);
    r->ib.y = v(J_INV_I_B + 3, J_SOFTNESS);
    r->ib.z = v(J_INV_I_B + 6, J_SOFTNESS + 1);
    if (r->info & JF_WELD) {
        r->axis = v(J_ANGULAR_IMPULSE, J_ANGULAR_IMPULSE);
        r->ia_ax = v(J_ANGULAR_MASS, J_ANGULAR_SPRING);
        r->ib_ax = v(J_ANGULAR_MASS + 3, J_ANGULAR_SPRING + 1);
        r->px = v(J_ANGULAR_MASS + 6, J_ANGULAR_SPRING + 2);
        r->s1 = s(pick(J_LINEAR_SPRING, J_LINEAR_SPRING + 1, J_LINEAR_SPRING + 2, J_LINEAR_SPRING));
        r->s2 = s(k == 0 ? J_LINEAR_HERTZ : J_ANGULAR_HERTZ);
        r->spring_imp = r->motor_imp = r->lower_imp = r->upper_imp = r->perp_x = r->perp_y = 0.0f;
    } else {
        int k3 = l3 ? 2 : k;
        r->axis = v(J_ROTATION_AXIS, J_ROTATION_AXIS);
        r->ia_ax = ldf(rec, JS_IAX + k3);
        r->ib_ax = ldf(rec, JS_IBX + k3);
        r->px = 0.0f;
        r->s1 = s(pick(J_SPRING_SOFTNESS, J_SPRING_SOFTNESS + 1, J_SPRING_SOFTNESS + 2, J_SOFTNESS + 2));
        r->s2 = s(pick(J_AXIAL_MASS, J_MAX_MOTOR_TORQUE, J_TARGET_ANGLE, J_MOTOR_SPEED));
        r->spring_imp = s(J_SPRING_IMPULSE);
        r->motor_imp = s(J_MOTOR_IMPULSE);
        r->lower_imp = s(J_LOWER_IMPULSE);
        r->upper_imp = s(J_UPPER_IMPULSE);
        r->perp_x = s(J_PERP_IMPULSE);
        r->perp_y = s(J_PERP_IMPULSE + 1);
    }
    jq_geometry(Q, r);
}

/* The row's scalars in all four lanes.  A wave with one joint keeps them
 * across the sweeps; with more it takes them out for each solve. */
struct JScal { Soft soft; float ma, mb, tw, relx, rely, kxx, kxy, kyy, kinv, axial, maxt, target, speed, lower, upper; QM ss; };
B3Q_FN void jq_scalars(const JQ& r, JScal* o) {
    o->soft = Soft{qbc<3>(r.ib.y), qbc<3>(r.ib.z), qbc<3>(r.s1)};
    o->ma = qbc<3>(r.ia.x);
    o->mb = qbc<3>(r.ib.x);
    o->lower = qbc<3>(r.ia.y);
    o->upper = qbc<3>(r.ia.z);
    o->tw = qbc<3>(r.ra);
    o->relx = qbc<3>(r.rb);
    o->rely = qbc<3>(r.psep);
    o->kxx = qbc<3>(r.px);
    o->kxy = qbc<3>(r.py);
    o->kyy = qbc<3>(r.pki.x);
    o->kinv = qbc<3>(r.pki.y);
    o->axial = qbc<0>(r.s2);
    o->maxt = qbc<1>(r.s2);
    o->target = qbc<2>(r.s2);
    o->speed = qbc<3>(r.s2);
    o->ss = QM{qbc<0>(r.s1), qbc<1>(r.s1), qbc<2>(r.s1)};
}

/* The joint's warm start (b3_warm_start_joints, 06:204-239), at the start of
 * the step: the anchors at the initial delta poses, the hinge rows as
 * b3_prepare_joints left them in the world. */
B3Q_FN void jq_warm(const QLane& Q, const JQ& r) {
    const Lane& L = Q.L;
    int k = Q.sub < 3 ? Q.sub : 2;
    float ang;
    if (ldi(L.w, jw(L, r.j, J_TYPE)) != kJointRevolute) {
        ang = ldf(L.w, jw(L, r.j, J_ANGULAR_IMPULSE + k));
    } else {
        float axial = r.spring_imp + r.motor_imp + r.lower_imp - r.upper_imp;
        float px = ldf(L.w, jw(L, r.j, J_PERP_X + k)), py = ldf(L.w, jw(L, r.j, J_PERP_Y + k));
        ang = px * r.perp_x + py * r.perp_y;
        ang = ang + axial * r.axis;
    }
    QVel x = qvel_load(Q, r.va, r.vb);
    x.va = x.va - qbc<3>(r.ia.x) * r.lin_imp;
    x.wa = x.wa - qmv(r.ia, qcross(r.ra, r.lin_imp) + ang);
    float dv = qbc<3>(r.ib.x) * r.lin_imp, dw = qmv(r.ib, qcross(r.rb, r.lin_imp) + ang);
    x.vb = x.vb + dv;
    x.wb = x.wb + dw;
    /* a joint of a body with itself: end b moves the body from where end a
     * left it (the solves take both ends from the same state, 06:204-239
     * against 06:436-642).  A wave without one skips it: as selects it cost
     * the chains 1 us of 151. */
    if (__ballot(r.va == r.vb) && r.va == r.vb) {
        x.vb = x.va + dv;
        x.wb = x.wa + dw;
    }
    qvel_store(Q, r.va, r.vb, r.info, x);
}

/* One joint's solve: b3_solve_revolute (06:436-642) or b3_solve_weld
 * (06:285-332), as solve_revolute and solve_weld. */
template <bool Bias>
B3Q_FN void jq_solve(const QLane& Q, JQ& r, const JScal& k, float h, float inv_h) {
    QVel x = qvel_load(Q, r.va, r.vb);
    const bool fixed = (r.info & JF_FIXED) != 0;
    Soft soft = k.soft;
    bool pbias = Bias;
    if (r.info & JF_WELD) {
        if (!fixed) {
            float bias = 0.0f, mscale = 1.0f, iscale = 0.0f;
            if (Bias || k.maxt > 0.0f) {
                bias = r.py * qbc<3>(r.ia_ax);
                mscale = qbc<3>(r.ib_ax);
                iscale = qbc<3>(r.px);
            }
            float cdot = x.wb - x.wa;
            float impulse = qmv(QM{r.ia_ax, r.ib_ax, r.px}, cdot + bias) * -mscale - iscale * r.axis;
            r.axis = r.axis + impulse;
            x.wa = x.wa - qmv(r.ia, impulse);
            x.wb = x.wb + qmv(r.ib, impulse);
        }
        pbias = Bias || k.axial > 0.0f;
        soft = Soft{k.ss.x, k.ss.y, k.ss.z};
    } else if (!fixed) {
        const float tw = k.tw, axial = k.axial, maxt = k.maxt, speed = k.speed, lower = k.lower, upper = k.upper;
        if (r.info & JF_SPRING) {
            float bias = k.ss.x * (tw - k.target);
            float cdot = qdot3(x.wb - x.wa, r.axis);
            float old = r.spring_imp;
            float dimp = -k.ss.y * axial * (cdot + bias) - k.ss.z * old;
            float nimp = old + dimp;
            if (maxt > 0.0f) {
                float maxp = maxt * h;
                nimp = clampf(nimp, -maxp, maxp);
            }
            dimp = nimp - old;
            r.spring_imp = nimp;
            x.wa = x.wa - dimp * r.ia_ax;
            x.wb = x.wb + dimp * r.ib_ax;
        }
        if (r.info & JF_MOTOR) {
            bool blocked = false;
            if (r.info & JF_LIMIT) {
                if (tw >= upper - 0.01f && speed > 0.0f) blocked = true;
                if (tw <= lower + 0.01f && speed < 0.0f) blocked = true;
            }
            if (blocked) {
                r.motor_imp = 0.0f;
            } else {
                float old = r.motor_imp;
                float cdot = qdot3(x.wb - x.wa, r.axis) - speed;
                float dimp = -axial * cdot;
                float nimp = old + dimp;
                float maxp = maxt * h;
                nimp = clampf(nimp, -maxp, maxp);
                dimp = nimp - old;
                r.motor_imp = nimp;
                x.wa = x.wa - dimp * r.ia_ax;
                x.wb = x.wb + dimp * r.ib_ax;
            }
        }
        if (r.info & JF_LIMIT) {
            float old = r.lower_imp;
            float lo = limit_impulse(tw - lower, qdot3(x.wb - x.wa, r.axis), inv_h, Bias, soft, axial, old);
            r.lower_imp = lo;
            float dimp = lo - old;
            x.wa = x.wa - dimp * r.ia_ax;
            x.wb = x.wb + dimp * r.ib_ax;
            old = r.upper_imp;
            float up = limit_impulse(upper - tw, qdot3(x.wa - x.wb, r.axis), inv_h, Bias, soft, axial, old);
            r.upper_imp = up;
            dimp = up - old;
            x.wa = x.wa + dimp * r.ia_ax;
            x.wb = x.wb - dimp * r.ib_ax;
        }
        V2 bias;
        bias.x = 0.0f;
        bias.y = 0.0f;
        float mscale = 1.0f, iscale = 0.0f;
        if (Bias) {
            bias.x = soft.bias_rate * k.relx;
            bias.y = soft.bias_rate * k.rely;
            mscale = soft.mass_scale;
            iscale = soft.impulse_scale;
        }
        float wrel = x.wb - x.wa;
        V2 rhs;
        rhs.x = qdot3(wrel, r.px) + bias.x;
        rhs.y = qdot3(wrel, r.py) + bias.y;
        V2 sol;
        sol.x = 0.0f;
        sol.y = 0.0f;
        if (k.kinv != kSingular) {
            sol.x = k.kinv * (k.kyy * rhs.x - k.kxy * rhs.y);
            sol.y = k.kinv * (-k.kxy * rhs.x + k.kxx * rhs.y);
        }
        V2 dimp;
        dimp.x = -mscale * sol.x - iscale * r.perp_x;
        dimp.y = -mscale * sol.y - iscale * r.perp_y;
        r.perp_x = r.perp_x + dimp.x;
        r.perp_y = r.perp_y + dimp.y;
        float ang = r.px * dimp.x + r.py * dimp.y;
        x.wa = x.wa - qmv(r.ia, ang);
        x.wb = x.wb + qmv(r.ib, ang);
    }
    /* the point rows (06:257-282) */
    float cdot = (x.vb + qcross(x.wb, r.rb)) - (x.va + qcross(x.wa, r.ra));
    float bias = 0.0f, mscale = 1.0f, iscale = 0.0f;
    if (pbias) {
        bias = r.psep * soft.bias_rate;
        mscale = soft.mass_scale;
        iscale = soft.impulse_scale;
    }
    float impulse = qmv(r.pki, cdot + bias) * -mscale - iscale * r.lin_imp;
    r.lin_imp = r.lin_imp + impulse;
    qimpulse(&x, k.ma, r.ia, k.mb, r.ib, r.ra, r.rb, impulse);
    qvel_store(Q, r.va, r.vb, r.info, x);
}

/* A row's impulses, and a hinge's latest perpendicular rows, to the world
 * (joint_writeback, joint_geometry). */
B3Q_FN void jq_writeback(const QLane& Q, const JQ& r) {
    const Lane& L = Q.L;
    uint32_t* w = L.w;
    auto put3 = [w, &L, &r, &Q](int f, float x) { if (Q.sub < 3) stf(w, jw(L, r.j, f + Q.sub), x); };
    auto put = [w, &L, &r, &Q](int f, float x) { if (Q.sub == 0) stf(w, jw(L, r.j, f), x); };
    put3(J_LINEAR_IMPULSE, r.lin_imp);
    if (r.info & JF_FIXED) return;
    if (r.info & JF_WELD) {
        put3(J_ANGULAR_IMPULSE, r.axis);
        return;
    }
    put3(J_PERP_X, r.px);
    put3(J_PERP_Y, r.py);
    put(J_PERP_IMPULSE, r.perp_x);
    put(J_PERP_IMPULSE + 1, r.perp_y);
    if (r.info & JF_SPRING) put(J_SPRING_IMPULSE, r.spring_imp);
    if (r.info & JF_MOTOR) put(J_MOTOR_IMPULSE, r.motor_imp);
    if (r.info & JF_LIMIT) {
        put(J_LOWER_IMPULSE, r.lower_imp);
        put(J_UPPER_IMPULSE, r.upper_imp);
    }
}

/* ---- force laws ---- */

/* A law of the force hook (b3d_lane.h) on quads: per-body rows of kWords LDS
 * words, staged once per step (stage), and each substep's velocity update of
 * bodies first, first + stride, ... (update; every worker stages and updates
 * the same bodies). */
struct QuadNoLaw {
    static constexpr int kWords = 0;
};

/* Plummer-softened gravity (GravityLaw, b3d_forces.h): body b's force is its
 * own sum over the other bodies in index order, the pairs (k, b), k < b,
 * subtracted and (b, j), j > b, added, which is the order in which the pair
 * loop reaches it; each pair's force is thus computed by both bodies'
 * workers, with the same operations.  Rows: center, mass, applied force,
 * inverse mass, gravity scale. */
struct QuadGravity {
    static constexpr int kWords = 9;
    float gravity, softening;
    const float* masses;   /* the world's, or null */

    static __device__ __attribute__((always_inline)) float* row(const QLane& Q, int b) {
        return lrow(Q, Q.q.law + b * kWords);
    }
    __device__ __attribute__((always_inline)) void stage(const QLane& Q, int nb) const {
        const Lane& L = Q.L;
        for (int b = Q.worker; b < nb; b += Q.workers) {
            V3 c = ld3(L.w, bw(L, b, B_CENTER)), f = ld3(L.w, bw(L, b, B_FORCE));
            float im = ldf(L.w, bw(L, b, B_INV_MASS)), gs = ldf(L.w, bw(L, b, B_GRAVITY_SCALE));
            int type = ldi(L.w, bw(L, b, B_TYPE));
            float m = masses ? masses[b] : (type == kDynamic && im > 0.0f ? 1.0f / im : 0.0f);
            float* r = row(Q, b);
            const float v[kWords] = {c.x, c.y, c.z, m, f.x, f.y, f.z, im, im > 0.0f ? gs : 0.0f};
#pragma unroll
            for (int k = 0; k < kWords; k++) r[k * kRow] = v[k];
        }
    }
    static __device__ __attribute__((always_inline)) V3 center(const QLane& Q, int b) {
        const float* r = row(Q, b);
        return add(v3(r[0], r[kRow], r[2 * kRow]), r3(delta_rec(Q.L, b), BD_DP));
    }
    __device__ __attribute__((always_inline)) void update(const QLane& Q, int nb, float h) const {
        const Lane& L = Q.L;
        float eps2 = softening * softening;
        V3 g = ld3(L.w, H_GRAVITY);
        for (int b = Q.worker; b < nb; b += Q.workers) {
            if (!(ru(delta_rec(L, b), BD_KIND) & kKindDynamic)) continue;
            const float* r = row(Q, b);
            float mb = r[3 * kRow], im = r[7 * kRow], gs = r[8 * kRow];
            V3 f = v3(r[4 * kRow], r[5 * kRow], r[6 * kRow]);
            V3 cb = center(Q, b);
            for (int k = 0; k < nb && mb != 0.0f; k++) {
                float mk = row(Q, k)[3 * kRow];
                if (k == b || mk == 0.0f) continue;
                bool before = k < b;
                V3 ck = center(Q, k);
                V3 d = before ? sub(cb, ck) : sub(ck, cb);
                float q = dot(d, d) + eps2;
                float inv = 1.0f / sqrtf(q);
                V3 p = scale(d, gravity * (before ? mk : mb) * (before ? mb : mk) * inv * inv * inv);
                f = before ? sub(f, p) : add(f, p);
            }
            const uint32_t* s = body_rec(L, b);
            V3 dv = add(scale(f, h * im), scale(g, h * gs));
            set_vlin(L, b, madd(dv, rf(s, BS_LD), vlin(L, b)));
            set_vang(L, b, madd(r3(s, BS_DW), rf(s, BS_AD), vang(L, b)));
        }
    }
};

/* ---- the step ---- */

/* The wave's contacts of one level: those in registers whose level it is,
 * then those past them in the order (pointer *at), loaded and stored. */
template <int CR, class Solve>
B3Q_FN void quad_level(const QLane& Q, CQ (&row)[CR], int cc, int lev, int* at, Solve solve) {
#pragma unroll
    for (int i = 0; i < CR; i++)
        if (row[i].lev == lev) solve(row[i]);
    while (*at < cc) {
        int e = lgeti(Q, Q.q.order + *at);
        if ((e >> 10) != lev) break;
        CQ r;
        cq_load(Q, e, &r);
        r.sep = cq_separations(Q, r, cq_base(Q, r));
        solve(r);
        cq_store(Q, r);
        *at += Q.waves;
    }
}

/* One b3_step (09_step.inl:148-264, default configuration) of the
 * workgroup's worlds.  Every thread runs it and meets every barrier; lanes
 * of worlds that do not step (L.active false) have no items.  `wg`: the
 * workgroup's words, zero at entry, as are the hit bits; a barrier has
 * passed since. */
template <int CR, int JR, class Law>
B3Q_FN void quad_step(QLane& Q, float dt, int substeps, int* wg, const Law& law) {
    Lane& L = Q.L;
    const bool act = L.active;
    int subs = substeps < 1 ? 1 : substeps;
    float h = dt / (float)subs;
    float inv_dt = 1.0f / dt;
    float inv_h = (float)subs * inv_dt;
    float hertz = minf(ldf(L.w, H_CONTACT_HERTZ), 0.25f * inv_h);
    float damping = ldf(L.w, H_CONTACT_DAMPING);
    Soft cs = make_soft(hertz, damping, h);
    Soft ss = make_soft(2.0f * hertz, 0.5f * damping, h);
    float contact_speed = ldf(L.w, H_CONTACT_SPEED);
    float rest_threshold = ldf(L.w, H_RESTITUTION_THRESHOLD);
    int old_n = act ? clampi(ldi(L.w, H_CONTACT_COUNT), 0, L.g.max_c) : 0;
    int ns = act ? clampi(ldi(L.w, H_SHAPE_COUNT), 0, L.g.max_s) : 0;
    count_bodies_and_joints(L);
    const int nb = L.nb, nj = L.nj;

    quad_open(Q, old_n, ns, nj);
    B3D_BARRIER();
    quad_overlaps(Q, ns);
    B3D_BARRIER();
    quad_collide(Q, ns, nj, old_n);
    B3D_BARRIER();
    int cc = 0;
    if (act) {
        cc = quad_append(Q, old_n, cs, ss, wg);
        body_prepass(L, h, Q.worker, Q.workers);
        if constexpr (Law::kWords > 0) law.stage(Q, nb);
        prepare_joints(L, h, Q.worker, Q.workers);
    }
    B3D_BARRIER();
    if (act) {
        if (Q.worker == 0) quad_levels(Q, cc, nb, wg);
        if (Q.worker == 4) quad_joint_levels(Q, nj, nb, wg);
        quad_joint_geometry<true>(Q, nj, 2);   /* the waves that build no levels */
    }
    B3D_BARRIER();
    const int nlev = __builtin_amdgcn_readfirstlane(wg[WG_LEVELS]);
    const int njlev = __builtin_amdgcn_readfirstlane(wg[WG_JLEVELS]);
    const int njmax = __builtin_amdgcn_readfirstlane(wg[WG_JOINTS]);
    const bool rest = __builtin_amdgcn_readfirstlane(wg[WG_REST]) != 0;
    CQ row[CR];
    float base[CR];
#pragma unroll
    for (int i = 0; i < CR; i++) {
        int at = i * Q.waves + Q.wave;
        row[i].c = -1;
        row[i].lev = 0;
        if (at < cc) {
            cq_load(Q, lgeti(Q, Q.q.order + at), &row[i]);
            base[i] = cq_base(Q, row[i]);
        }
    }
    JQ joint[JR];
#pragma unroll
    for (int i = 0; i < JR; i++) {
        int j = i * Q.waves + Q.wave;
        joint[i].j = -1;
        joint[i].lev = 0;
        if (j < nj) jq_load(Q, j, &joint[i]);
    }
    const int past = CR * Q.waves + Q.wave;   /* the wave's first contact not in registers */
    auto levels = [&](auto solve) {
        int at = past;
        for (int lev = 1; lev <= nlev; lev++) {
            quad_level<CR>(Q, row, cc, lev, &at, solve);
            B3D_BARRIER();
        }
    };
    JScal scal;
    if (JR == 1 && joint[0].j >= 0) jq_scalars(joint[0], &scal);
    auto joint_levels = [&](auto solve) {
        for (int lev = 1; lev <= njlev; lev++) {
#pragma unroll
            for (int i = 0; i < JR; i++)
                if ((joint[i].lev & 255) == lev || (joint[i].lev >> 8) == lev) {
                    if (JR > 1) jq_scalars(joint[i], &scal);
                    solve(joint[i], scal);
                }
            B3D_BARRIER();
        }
    };
    auto separations = [&]() {
#pragma unroll
        for (int i = 0; i < CR; i++)
            if (row[i].lev > 0) row[i].sep = cq_separations(Q, row[i], base[i]);
    };
    separations();
    levels([&](CQ& r) { cq_warm(Q, r); });
    for (int j = 0; j < njmax; j++) {
#pragma unroll
        for (int i = 0; i < JR; i++)
            if (joint[i].j == j) jq_warm(Q, joint[i]);
        B3D_BARRIER();
    }
    for (int s = 0; s < subs; s++) {
        if (act) {
            if constexpr (Law::kWords > 0) law.update(Q, nb, h);
            else integrate_velocities(L, Q.worker, Q.workers);
        }
        B3D_BARRIER();
        levels([&](CQ& r) { cq_solve<false>(Q, r, inv_h, contact_speed, cs, ss); });
        joint_levels([&](JQ& r, const JScal& k) { jq_solve<true>(Q, r, k, h, inv_h); });
        if (act) integrate_positions(L, h, inv_dt, Q.worker, Q.workers);
        B3D_BARRIER();
        if (njmax > 0) {
            quad_joint_geometry<false>(Q, nj, 0);
            B3D_BARRIER();
#pragma unroll
            for (int i = 0; i < JR; i++)
                if (joint[i].j >= 0) jq_geometry(Q, &joint[i]);
            if (JR == 1 && joint[0].j >= 0) jq_scalars(joint[0], &scal);
        }
        separations();
        levels([&](CQ& r) { cq_solve<true>(Q, r, inv_h, contact_speed, cs, ss); });
        joint_levels([&](JQ& r, const JScal& k) { jq_solve<false>(Q, r, k, h, inv_h); });
        if (rest) levels([&](CQ& r) { cq_restitution(Q, r, rest_threshold); });
    }
#pragma unroll
    for (int i = 0; i < CR; i++)
        if (row[i].lev > 0) cq_writeback(Q, row[i]);
    for (int at = past; at < cc; at += Q.waves) {
        CQ r;
        cq_load(Q, lgeti(Q, Q.q.order + at), &r);
        cq_writeback(Q, r);
    }
#pragma unroll
    for (int i = 0; i < JR; i++)
        if (joint[i].j >= 0) jq_writeback(Q, joint[i]);
    if (act) {
        finalize(L, Q.worker, Q.workers);
        vel_store(L, Q.worker, Q.workers);
    }
}

/* The view of one lane of a workgroup of `waves` waves: world `slot` of a
 * tile, its words at w, the tile's scratch (scratch_tile_words) and stage. */
B3Q_FN QLane quad_lane(uint32_t* w, uint32_t* tile_scratch, uint32_t* tile_stage, float* lds, const Geometry& g,
        const QuadLayout& q, int slot, int waves, unsigned int opts) {
    QLane Q;
    Q.sub = (int)(threadIdx.x & 3u);
    Q.wave = (int)(threadIdx.x >> 6);
    Q.worker = Q.wave * 4 + Q.sub;
    Q.waves = waves;
    Q.workers = 4 * waves;
    Q.q = q;
    Q.lds = lds + kQuadWgWords + slot % kQuadCols;
    Q.recs = tile_scratch + (size_t)g.scr_words * kLanes + (size_t)slot * g.max_c * kQRecWords;
    Q.st = PairStage{};
    Q.st.p = tile_stage + slot;
    Q.L = lane_view(nullptr, nullptr, nullptr, g, 0, slot, opts);
    Q.L.w = w;
    Q.L.scr = tile_scratch + (size_t)slot * (kWord == kLanes ? 1 : g.scr_words);
    Q.L.sq = reinterpret_cast<uint32_t*>(Q.lds);
    Q.L.vel = Q.lds + q.y * kRow;
    return Q;
}
/* Clears what quad_step expects cleared; a barrier follows. */
B3Q_FN void quad_clear(const QLane& Q, int* wg) {
    if (threadIdx.x < (unsigned)kQuadWgWords) wg[threadIdx.x] = 0;
    for (int k = Q.worker; k <= hit_words(Q.L.g); k += Q.workers) lseti(Q, Q.q.hits + k, 0);
}

}  // namespace b3d

#endif
