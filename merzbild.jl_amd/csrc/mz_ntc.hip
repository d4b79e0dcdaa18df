// mz_ntc.hip -- NTC pair selection with VHS collisions on gfx950.
//
// Reference (Merzbild.jl, src/collisions/):
//   compute_n_coll_*                collision_ntc.jl:173-197
//   collide_2particles_vhs!         collision_ntc.jl:223-270
//   collide_2particles_vhs_equal_weight!  collision_ntc.jl:294-309
//   ntc! / ntc_equal_weight!        collision_ntc.jl:338-595
//   compute_com!, compute_g!        collision_utils.jl:374-391
//   scatter_vhs!                    collision_scattering.jl:17-29
//   sigma_vhs                       collision_cross_sections.jl:179-181
//
// The candidate loop of one cell is sequential in the reference: the running
// (sigma g w)_max is updated before every acceptance test, and particles
// created by a split become candidates of the same loop.  Cells run in
// parallel, a cell with several candidates on a wavefront that evaluates them
// ahead (ntc_windows), other cells and replayed draws one lane each.  Draw
// order per cell stream:
// [n_coll], then per candidate [i, k (, k redraws)], [accept] if g > eps,
// [phi, cos theta] if accepted.
//
// Particle creation (weight splitting) follows the reference's append at the
// global end: created particles are first written to per-cell scratch (the
// loop sees them as group-2 members), then appended in cell order, which is
// the order a sequential loop over cells produces; ids come from the emulated
// free-id LIFO, growing `length` by DELTA_PARTICLES when it runs dry, as
// resize! does (src/particles.jl:269-298, 311-332, 426-433).
#include "mz_phys.h"

#include <algorithm>
#include <cstring>
#include <vector>

struct NtcArgs {
    MzSpView a, b;       // species s1, s2 (same view when s1 == s2)
    int32_t single;      // s1 == s2
    int32_t equal_weight;
    int32_t may_split;
    int32_t cell_lo, cell_hi;  // 0-based inclusive
    double dt, dw_tol;
    double mu1, mu2, factor, expo;
    const double *V;
    double *sgwm;        // [n_cells] of this pair
    int32_t *cnt;        // [n_cells][5]
    MzRngParams rp;
    // split path
    const int32_t *ncoll_in;   // [n_cells] from the count pass (NULL: draw here)
    const int64_t *soff;       // [n_cells] scratch offsets
    double *sc[7];             // scratch SoA: x0 x1 x2 v0 v1 v2 w, per species half
    int64_t sc_cap;            // entries per species half
    int32_t *created;          // [2][n_cells]
};

__device__ inline int64_t slot_of(const MzSpView &sp, int c, int32_t li, int32_t n1, int32_t n2) {
    // map_cont_index (src/particles.jl:364-366) for positions present before the call
    return li < n1 ? (int64_t)sp.pia.start1[c] - 1 + li : (int64_t)sp.pia.start2[c] - 1 + (li - n1);
}

// Particle handle: either a slot of the store or a scratch entry.
struct PRef {
    double *x0, *x1, *x2, *v0, *v1, *v2, *w;
    int64_t i;
};

__device__ inline PRef pref_slot(const MzSpView &sp, int64_t p) {
    return PRef{sp.x0, sp.x1, sp.x2, sp.v0, sp.v1, sp.v2, sp.w, p};
}

__device__ inline PRef pref_scratch(const NtcArgs &A, int half, int64_t e) {
    int64_t o = (int64_t)half * A.sc_cap;
    return PRef{A.sc[0] + o, A.sc[1] + o, A.sc[2] + o, A.sc[3] + o, A.sc[4] + o, A.sc[5] + o, A.sc[6] + o, e};
}

// A cell's fixed values and the candidate loop's running state.
struct NtcCell {
    int32_t n1a, n2a, n1b, n2b, nla, nlb;
    int64_t s_base, n_coll;
};
struct NtcState {
    int32_t na, nb;       // current n_local (grows with splits)
    int32_t ca, cb;       // created per species
    int32_t performed, eqw;
    double sgwm;
};

// Particle i of species half 0 (k of half 1) of cell c: a position present
// before the call or this call's scratch entry.
__device__ inline PRef ntc_ref_a(const NtcArgs &A, int c, const NtcCell &C, int32_t i) {
    return i < C.nla ? pref_slot(A.a, slot_of(A.a, c, i, C.n1a, C.n2a)) : pref_scratch(A, 0, C.s_base + (i - C.nla));
}
__device__ inline PRef ntc_ref_b(const NtcArgs &A, int c, const NtcCell &C, int32_t k) {
    return k < C.nlb ? pref_slot(A.b, slot_of(A.b, c, k, C.n1b, C.n2b)) : pref_scratch(A, 1, C.s_base + (k - C.nlb));
}

// A cell's setup: counts, (sigma g w)_max and n_coll (draw 0 of its stream,
// or the count pass's value).
template <class Draw>
__device__ __forceinline__ void ntc_setup(const NtcArgs &A, const int c, Draw &dr, NtcCell &C, NtcState &S) {
    C.n1a = A.a.pia.n1[c]; C.n2a = A.a.pia.n2[c];
    C.n1b = A.b.pia.n1[c]; C.n2b = A.b.pia.n2[c];
    C.nla = A.a.pia.nloc[c]; C.nlb = A.b.pia.nloc[c];
    S.sgwm = A.sgwm[c];
    int64_t n_coll;
    if (A.ncoll_in) {
        n_coll = A.ncoll_in[c];
        dr.seek(1);
    } else {
        double R = dr.next();
        n_coll = (int64_t)floor(mz_ncoll_est(A.single, A.dt, C.nla, C.nlb, S.sgwm, A.V[c], R));
    }
    if (!(n_coll <= MZ_NTC_MAX_CANDIDATES)) {   // also catches NaN estimates
        atomicOr(&A.a.ctr->err, MZ_ERR_SCRATCH);
        n_coll = 0;
    }
    C.n_coll = n_coll;
    S.na = C.nla; S.nb = C.nlb;
    S.ca = 0; S.cb = 0;
    S.performed = 0; S.eqw = 0;
    C.s_base = A.may_split ? A.soff[c] : 0;
}

// Whether this call's scratch has room for the split a collision of the
// pair makes (always true when it makes none).  Without room the scratch
// error is raised and the candidate ends before its scattering draws, as a
// performed collision.
__device__ inline bool ntc_split_room(const NtcArgs &A, const NtcCell &C, const NtcState &S, double wi, double wk) {
    if (A.equal_weight || fabs(wi - wk) < A.dw_tol || !A.may_split) return true;
    const bool on_a = wi > wk || A.single;
    const int32_t q = on_a ? (A.single ? S.ca + S.cb : S.ca) : S.cb;
    if (q < C.n_coll) return true;
    atomicOr(&(on_a ? A.a : A.b).ctr->err, MZ_ERR_SCRATCH);
    return false;
}

// The collision of a pair that passed the acceptance test, with room for
// its split (collide_2particles_vhs! with weight splitting,
// collision_ntc.jl:223-270): the split (the heavier particle leaves a copy of
// itself with the weight difference and takes the lighter's weight), then
// the post-collision velocities u.
__device__ __forceinline__ void ntc_collide(const NtcArgs &A, const NtcCell &C, NtcState &S, const PRef &pi,
                                            const PRef &pk, double vi0, double vi1, double vi2, double vk0,
                                            double vk1, double vk2, double wi, double wk, double ui0, double ui1,
                                            double ui2, double uk0, double uk1, double uk2) {
    ++S.performed;
    if (A.equal_weight || fabs(wi - wk) < A.dw_tol) {
        ++S.eqw;
    } else if (!A.may_split) {
        atomicOr(&A.a.ctr->err, MZ_ERR_SCRATCH);
    } else if (wi > wk) {
        PRef nw = pref_scratch(A, 0, C.s_base + (A.single ? S.ca + S.cb : S.ca));
        nw.x0[nw.i] = pi.x0[pi.i]; nw.x1[nw.i] = pi.x1[pi.i]; nw.x2[nw.i] = pi.x2[pi.i];
        nw.v0[nw.i] = vi0; nw.v1[nw.i] = vi1; nw.v2[nw.i] = vi2;
        nw.w[nw.i] = wi - wk;
        pi.w[pi.i] = wk;
        ++S.ca; ++S.na;
    } else if (A.single) {
        PRef nw = pref_scratch(A, 0, C.s_base + S.ca + S.cb);
        nw.x0[nw.i] = pk.x0[pk.i]; nw.x1[nw.i] = pk.x1[pk.i]; nw.x2[nw.i] = pk.x2[pk.i];
        nw.v0[nw.i] = vk0; nw.v1[nw.i] = vk1; nw.v2[nw.i] = vk2;
        nw.w[nw.i] = wk - wi;
        pk.w[pk.i] = wi;
        ++S.ca; ++S.na;
    } else {
        PRef nw = pref_scratch(A, 1, C.s_base + S.cb);
        nw.x0[nw.i] = pk.x0[pk.i]; nw.x1[nw.i] = pk.x1[pk.i]; nw.x2[nw.i] = pk.x2[pk.i];
        nw.v0[nw.i] = vk0; nw.v1[nw.i] = vk1; nw.v2[nw.i] = vk2;
        nw.w[nw.i] = wk - wi;
        pk.w[pk.i] = wi;
        ++S.cb; ++S.nb;
    }
    pi.v0[pi.i] = ui0; pi.v1[pi.i] = ui1; pi.v2[pi.i] = ui2;
    pk.v0[pk.i] = uk0; pk.v1[pk.i] = uk1; pk.v2[pk.i] = uk2;
}

// One candidate of cell c's loop (collision_ntc.jl:338-380); false when a
// replay row ran out.
template <class Draw>
__device__ __forceinline__ bool ntc_candidate(const NtcArgs &A, const int c, const NtcCell &C, NtcState &S,
                                              Draw &dr) {
    int32_t i = (int32_t)floor(dr.next() * (double)S.na);
    int32_t k = (int32_t)floor(dr.next() * (double)(A.single ? S.na : S.nb));
    if (A.single) {
        while (i == k) {
            k = (int32_t)floor(dr.next() * (double)S.na);
            if (dr.exhausted()) return false;   // replay row exhausted
        }
    }
    const PRef pi = ntc_ref_a(A, c, C, i);
    const PRef pk = A.single ? ntc_ref_a(A, c, C, k) : ntc_ref_b(A, c, C, k);
    const double vi0 = pi.v0[pi.i], vi1 = pi.v1[pi.i], vi2 = pi.v2[pi.i];
    const double vk0 = pk.v0[pk.i], vk1 = pk.v1[pk.i], vk2 = pk.v2[pk.i];
    double g0, g1, g2;
    const double g = mz_rel_speed(vi0, vi1, vi2, vk0, vk1, vk2, g0, g1, g2);
    if (!(g > MZ_G_EPS)) return true;
    const double wi = pi.w[pi.i], wk = pk.w[pk.i];
    const double sgw = mz_vhs_sgw(A.factor, A.expo, g, wi, wk);
    S.sgwm = sgw > S.sgwm ? sgw : S.sgwm;
    if (!(dr.next() < sgw / S.sgwm)) return true;
    if (!ntc_split_room(A, C, S, wi, wk)) {
        ++S.performed;
        return true;
    }
    double vc0, vc1, vc2;
    mz_com(A.mu1, A.mu2, vi0, vi1, vi2, vk0, vk1, vk2, vc0, vc1, vc2);
    // scatter_vhs!: phi first, then cos(theta)
    const double R_phi = dr.next();
    const double R_ct = dr.next();
    double ui0, ui1, ui2, uk0, uk1, uk2;
    mz_vhs_post(A.mu1, A.mu2, g, vc0, vc1, vc2, R_phi, R_ct, ui0, ui1, ui2, uk0, uk1, uk2);
    ntc_collide(A, C, S, pi, pk, vi0, vi1, vi2, vk0, vk1, vk2, wi, wk, ui0, ui1, ui2, uk0, uk1, uk2);
    return true;
}

// One candidate of cell c's swpm! loop (collision_swpm.jl:201-288); false
// when a replay row ran out.  S.sgwm is (sigma g)_max, S.ca the created.
template <class Draw>
__device__ __forceinline__ bool swpm_candidate(const NtcArgs &A, const int c, const NtcCell &C, NtcState &S, Draw &dr,
                                               const double wtf, const double inv_w_max) {
    const int32_t i = (int32_t)floor(dr.next() * (double)S.na);
    int32_t k = (int32_t)floor(dr.next() * (double)S.na);
    while (i == k) {
        k = (int32_t)floor(dr.next() * (double)S.na);
        if (dr.exhausted()) return false;   // replay row exhausted
    }
    const PRef pi = ntc_ref_a(A, c, C, i), pk = ntc_ref_a(A, c, C, k);
    const double vi0 = pi.v0[pi.i], vi1 = pi.v1[pi.i], vi2 = pi.v2[pi.i];
    const double vk0 = pk.v0[pk.i], vk1 = pk.v1[pk.i], vk2 = pk.v2[pk.i];
    double g0, g1, g2;
    const double g = mz_rel_speed(vi0, vi1, vi2, vk0, vk1, vk2, g0, g1, g2);
    if (!(g > MZ_G_EPS)) return true;
    const double sgm = mz_vhs_sgw(A.factor, A.expo, g, 1.0, 1.0);   // sigma g
    S.sgwm = sgm > S.sgwm ? sgm : S.sgwm;
    const double wi = pi.w[pi.i], wk = pk.w[pk.i];
    if (!(dr.next() < sgm * (wi > wk ? wi : wk) * inv_w_max / S.sgwm)) return true;
    ++S.performed;
    double vc0, vc1, vc2;
    mz_com(A.mu1, A.mu2, vi0, vi1, vi2, vk0, vk1, vk2, vc0, vc1, vc2);
    const double dw = (wi < wk ? wi : wk) * wtf;
    pi.w[pi.i] = wi - dw;
    pk.w[pk.i] = wk - dw;
    if (S.ca + 1 >= 2 * C.n_coll) {
        atomicOr(&A.a.ctr->err, MZ_ERR_SCRATCH);
        return true;
    }
    const PRef n_i = pref_scratch(A, 0, C.s_base + S.ca), n_k = pref_scratch(A, 0, C.s_base + S.ca + 1);
    n_i.x0[n_i.i] = pi.x0[pi.i]; n_i.x1[n_i.i] = pi.x1[pi.i]; n_i.x2[n_i.i] = pi.x2[pi.i];
    n_k.x0[n_k.i] = pk.x0[pk.i]; n_k.x1[n_k.i] = pk.x1[pk.i]; n_k.x2[n_k.i] = pk.x2[pk.i];
    n_i.w[n_i.i] = dw;
    n_k.w[n_k.i] = dw;
    S.ca += 2;
    S.na += 2;
    // scatter_vhs! on the two new particles: phi first, then cos(theta)
    const double R_phi = dr.next();
    const double R_ct = dr.next();
    double ui0, ui1, ui2, uk0, uk1, uk2;
    mz_vhs_post(A.mu1, A.mu2, g, vc0, vc1, vc2, R_phi, R_ct, ui0, ui1, ui2, uk0, uk1, uk2);
    n_i.v0[n_i.i] = ui0; n_i.v1[n_i.i] = ui1; n_i.v2[n_i.i] = ui2;
    n_k.v0[n_k.i] = uk0; n_k.v1[n_k.i] = uk1; n_k.v2[n_k.i] = uk2;
    return true;
}

// The end of a cell's loop: (sigma g w)_max, the counters, created counts.
__device__ __forceinline__ void ntc_finish_cell(const NtcArgs &A, const int c, const NtcCell &C,
                                                const NtcState &S) {
    A.sgwm[c] = S.sgwm;
    int32_t *cn = A.cnt + (int64_t)c * 5;
    cn[0] = C.nla;
    cn[1] = A.single ? C.nla : C.nlb;
    cn[2] = (int32_t)C.n_coll;
    cn[3] = S.performed;
    cn[4] = S.eqw;
    if (A.may_split) {
        A.created[c] = A.single ? S.ca + S.cb : S.ca;
        A.created[(int64_t)(A.cell_hi + 1) + c] = A.single ? 0 : S.cb;
    }
}

// Draws of a cell's stream for one lane: mz_rand.
struct NtcLaneDraw {
    const MzRngParams &rp;
    MzStream st;
    __device__ double next() { return mz_rand(rp, st); }
    __device__ bool exhausted() const { return rp.mode == 1 && (int64_t)st.k > rp.cols; }
    __device__ void seek(uint64_t k) { st.k = k; }
};

// Draws of a cell's stream for a whole wavefront running the cell (Philox
// draws only): lane L holds Philox block base / 2 + L, i.e. draws base + 2 L
// and base + 2 L + 1, and every lane reads draw k from its lane; the block
// of 128 draws is computed again, all lanes at once, when k leaves it.
struct NtcWaveDraw {
    const MzRngParams &rp;
    uint64_t stream, k, base;
    double h0, h1;
    __device__ double next() {
        const uint64_t kk = k++;
        if (kk < base || kk >= base + 128) {
            base = kk & ~(uint64_t)1;
            mz_philox_pair(rp, stream, (base >> 1) + (uint64_t)(threadIdx.x & 63), h0, h1);
        }
        const uint64_t idx = kk - base;
        const int l = (int)(idx >> 1);
        const double a = mz_readlane_d(h0, l), b = mz_readlane_d(h1, l);
        return (idx & 1) ? b : a;
    }
    __device__ bool exhausted() const { return false; }
    __device__ void seek(uint64_t kk) { k = kk; }
    // the block holds draws D .. D + span - 1 afterwards (span <= 127)
    __device__ void cover(uint64_t D, int span) {
        if (D < base || D + (uint64_t)span > base + 128) {
            base = D & ~(uint64_t)1;
            mz_philox_pair(rp, stream, (base >> 1) + (uint64_t)(threadIdx.x & 63), h0, h1);
        }
    }
    // draw base + idx for this lane (idx may differ between lanes; idx < 128)
    __device__ double at(int idx) const {
        const int l = idx >> 1;
        const double a = __shfl(h0, l, 64), b = __shfl(h1, l, 64);
        return (idx & 1) ? b : a;
    }
};

// A cell's candidate loop on a whole wavefront (Philox draws), candidates
// evaluated ahead.  A candidate that is rejected takes three draws and one
// that collides takes five, and a collision of unequal weights adds a known
// number of particles to the cell, so the candidate reached after `a`
// collisions and `r` rejections of a window that starts at draw D begins at
// draw D + 5 a + 3 r and picks from na0 + inc a particles.  A window
// evaluates that lattice: lane a M + j takes the candidate after a
// collisions and j rejections (T tracks of M candidates, T M <= 64) -- pair,
// relative speed, collision rate, acceptance test, post-collision
// velocities.  The wave then follows the sequential loop's path through it
// (mz_window_walk): a new (sigma g w)_max renews every lane's acceptance
// test, and the window ends, and the next one starts at that draw, at a
// candidate that shares a particle with a collision of the window or picks
// one created in it, where the particle count is not the predicted one, and
// where a track or the tracks run out; then all its collisions are carried
// out at once.  T follows the acceptance rate (doubled when the tracks run
// out, halved when a track does).  A candidate whose k must be drawn again
// runs on its own.  Same draws, same operands, same order of updates as the
// loop over ntc_candidate: the results are equal.
//
// What bounds it: the latency of one window (draw exchange, the two gathers,
// the power chain; about 4 us) times the windows of the cell with the most.
// Few acceptances make windows of 40 candidates, many make eight tracks of
// eight.  Measured against one lane per cell, and (the last two) against windows
// that ended at every split, in states of 50 passes and more: 8,192 boxes of 90
// particles with 130 candidates, 8% accepted, 4,030 -> 310 us a call; 2,048 boxes
// with 580 candidates (up to 3,500), 4% accepted, SWPM, 5,560 -> 270 us; 4,096
// boxes with 150 candidates, 39% accepted, SWPM, 1,220 -> 270 us; 1,024 cells of up
// to 30,000 particles, 290 candidates (up to 2,900), 40% accepted, 3,250 -> 710 us;
// 500 cells of 35 candidates, 5% accepted, 46 -> 19 us.
#define NTC_T1_LEN 40   // candidates of a single track (its draws fit the 128 held)

enum { NTC_PLAIN = 0, NTC_SPLIT = 1, NTC_SWPM = 2 };   // no particles created; ntc! with splitting; swpm!

template <int KIND>
__device__ __forceinline__ void ntc_windows(const NtcArgs &A, const int c, const NtcCell &C, NtcState &S,
                                            NtcWaveDraw &dr, const double wtf, const double inv_w_max) {
    constexpr bool SWPM = KIND == NTC_SWPM, CREATES = KIND != NTC_PLAIN;
    const int lane = threadIdx.x & 63;
    const bool single = SWPM || A.single;
    const int32_t st1a = A.a.pia.start1[c] - 1, st2a = A.a.pia.start2[c] - 1;
    const int32_t st1b = A.b.pia.start1[c] - 1, st2b = A.b.pia.start2[c] - 1;
    const int64_t sc_b = !CREATES || single ? 0 : A.sc_cap;   // species half 1 of the scratch
    int lt = 2;   // log2 of the number of tracks T: 0 .. 3
    int32_t inc = SWPM ? 2 : (CREATES && single ? 1 : 0);
    int64_t cc = 0;
    uint64_t o = dr.k;
    while (cc < C.n_coll) {
        const uint64_t D = o;
        const int T = 1 << lt, M = lt == 0 ? NTC_T1_LEN : 64 >> lt;
        dr.cover(D, 5 * (T - 1) + 3 * (M - 1) + 5);
        const int32_t na0 = S.na, nb0 = single ? S.na : S.nb;
        const int a_l = lt == 0 ? 0 : lane >> (6 - lt);
        const int j_l = lane - a_l * M;
        const int64_t cand = cc + a_l + j_l;
        const bool live = j_l < M && cand < C.n_coll;
        const int idx = min((int)(D - dr.base) + 5 * a_l + 3 * j_l, 123);
        const double d0 = dr.at(idx), d1 = dr.at(idx + 1), d2 = dr.at(idx + 2), d3 = dr.at(idx + 3),
                     d4 = dr.at(idx + 4);
        const int32_t si = (int32_t)floor(d0 * (double)(na0 + inc * a_l));
        const int32_t sk = (int32_t)floor(d1 * (double)(nb0 + inc * a_l));
        const bool fresh = si >= na0 || sk >= nb0;   // created in this window (or out of range by rounding)
        const bool same = single && si == sk;
        bool slow = false;                            // g <= eps: no acceptance draw
        double vi0 = 0.0, vi1 = 0.0, vi2 = 0.0, vk0 = 0.0, vk1 = 0.0, vk2 = 0.0, wi = 0.0, wk = 0.0;
        double sg = 0.0, t = 0.0;                     // rate entering the running maximum; acceptance numerator
        double ui0 = 0.0, ui1 = 0.0, ui2 = 0.0, uk0 = 0.0, uk1 = 0.0, uk2 = 0.0;
        double xi0 = 0.0, xi1 = 0.0, xi2 = 0.0, xk0 = 0.0, xk1 = 0.0, xk2 = 0.0;
        const bool in_i = !CREATES || si < C.nla, in_k = !CREATES || sk < C.nlb;
        const int64_t pi = in_i ? (int64_t)(si < C.n1a ? st1a + si : st2a + (si - C.n1a)) : C.s_base + (si - C.nla);
        const int64_t pk = in_k ? (int64_t)(sk < C.n1b ? st1b + sk : st2b + (sk - C.n1b))
                                : sc_b + C.s_base + (sk - C.nlb);
        double sgwm = S.sgwm;
        bool acc = false, eq = KIND == NTC_PLAIN;     // eq: the collision makes no split
        if (live && !fresh && !same) {
            vi0 = (in_i ? A.a.v0 : A.sc[3])[pi]; vk0 = (in_k ? A.b.v0 : A.sc[3])[pk];
            vi1 = (in_i ? A.a.v1 : A.sc[4])[pi]; vk1 = (in_k ? A.b.v1 : A.sc[4])[pk];
            vi2 = (in_i ? A.a.v2 : A.sc[5])[pi]; vk2 = (in_k ? A.b.v2 : A.sc[5])[pk];
            wi = (in_i ? A.a.w : A.sc[6])[pi];
            wk = (in_k ? A.b.w : A.sc[6])[pk];
            if (KIND == NTC_SPLIT) eq = fabs(wi - wk) < A.dw_tol;
            // the direction needs the draws only: it is worked out while the
            // loads are in flight, for every candidate
            double e0, e1, e2;
            mz_vhs_dir(d3, d4, e0, e1, e2);
            double g0, g1, g2;
            const double g = mz_rel_speed(vi0, vi1, vi2, vk0, vk1, vk2, g0, g1, g2);
            slow = !(g > MZ_G_EPS);
            if (SWPM) {
                sg = mz_vhs_sgw(A.factor, A.expo, g, 1.0, 1.0);
                t = sg * (wi > wk ? wi : wk) * inv_w_max;
            } else {
                sg = mz_vhs_sgw(A.factor, A.expo, g, wi, wk);
                t = sg;
            }
            // every candidate that can be accepted: a larger maximum only
            // lowers t / (sigma g w)_max
            acc = d2 < t / sgwm;
            if (acc) {
                // the particle that a split copies: the heavier, or the
                // second of two equal ones that dw_tol does not call equal
                if (SWPM || (CREATES && !eq && wi > wk)) {
                    xi0 = (in_i ? A.a.x0 : A.sc[0])[pi]; xi1 = (in_i ? A.a.x1 : A.sc[1])[pi];
                    xi2 = (in_i ? A.a.x2 : A.sc[2])[pi];
                }
                if (SWPM || (CREATES && !eq && !(wi > wk))) {
                    xk0 = (in_k ? A.b.x0 : A.sc[0])[pk]; xk1 = (in_k ? A.b.x1 : A.sc[1])[pk];
                    xk2 = (in_k ? A.b.x2 : A.sc[2])[pk];
                }
                double vc0, vc1, vc2;
                mz_com(A.mu1, A.mu2, vi0, vi1, vi2, vk0, vk1, vk2, vc0, vc1, vc2);
                mz_vhs_along(A.mu1, A.mu2, g, vc0, vc1, vc2, e0, e1, e2, ui0, ui1, ui2, uk0, uk1, uk2);
            }
        }
        const uint64_t samem = __ballot(live && same && !fresh), slowm = __ballot(slow);
        const uint64_t stop = __ballot(!live || fresh) | samem | slowm, ends = mz_window_ends(lt, NTC_T1_LEN);
        // collisions after which the particle count is not the predicted one
        const uint64_t eqm = __ballot(eq), last = KIND != NTC_SPLIT ? 0 : __ballot(eq == (inc > 0));
        uint64_t accm = __ballot(acc), maxm = __ballot(sg > sgwm);
        uint64_t taken = 0, seen = 0, dirty = 0, checked = 0;
        int pos = 0, why;
        for (;;) {
            why = mz_window_walk(accm, stop | maxm, last, ends, T * M, M, pos, taken, seen);
            // candidates that share a particle with an earlier collision
            for (uint64_t m = taken & ~checked; m; m &= m - 1) {
                const int L = __builtin_ctzll(m);
                const int32_t i = __builtin_amdgcn_readlane(si, L), k = __builtin_amdgcn_readlane(sk, L);
                dirty |= __ballot(single ? si == i || sk == i || si == k || sk == k : si == i || sk == k) &
                         (~1ull << L);
            }
            checked = taken;
            if (dirty & seen) {
                pos = __builtin_ctzll(dirty & seen);
                taken &= (1ull << pos) - 1;
                why = -1;
                break;
            }
            if (why != MZ_WALK_STOP || (stop >> pos) & 1) break;
            sgwm = mz_readlane_d(sg, pos);   // above the running maximum
            accm = __ballot(acc && d2 < t / sgwm);
            maxm = __ballot(sg > sgwm);
        }
        const int a = __popcll(taken), j = pos - a * M;
        // The window's collisions, all at once: no particle is in two of them.
        // Each makes at most one split (SWPM: two particles), so the scratch,
        // one entry (two) per candidate, has room.
        const bool heavy_i = wi > wk;
        const bool on_a = KIND != NTC_SPLIT || single || heavy_i;
        if ((taken >> lane) & 1) {
            if (SWPM) {
                const double dw = (wi < wk ? wi : wk) * wtf;
                (in_i ? A.a.w : A.sc[6])[pi] = wi - dw;
                (in_k ? A.b.w : A.sc[6])[pk] = wk - dw;
                const int64_t e = C.s_base + S.ca + 2 * __popcll(taken & mz_lanemask_lt());
                A.sc[0][e] = xi0; A.sc[1][e] = xi1; A.sc[2][e] = xi2;
                A.sc[3][e] = ui0; A.sc[4][e] = ui1; A.sc[5][e] = ui2; A.sc[6][e] = dw;
                A.sc[0][e + 1] = xk0; A.sc[1][e + 1] = xk1; A.sc[2][e + 1] = xk2;
                A.sc[3][e + 1] = uk0; A.sc[4][e + 1] = uk1; A.sc[5][e + 1] = uk2; A.sc[6][e + 1] = dw;
            } else {
                if (KIND == NTC_SPLIT && !eq) {
                    // the split of the heavier particle
                    const int32_t q = (on_a ? (single ? S.ca + S.cb : S.ca) : S.cb) +
                                      __popcll(taken & ~eqm & mz_lanemask_lt());
                    const int64_t e = (on_a ? 0 : sc_b) + C.s_base + q;
                    A.sc[0][e] = heavy_i ? xi0 : xk0; A.sc[1][e] = heavy_i ? xi1 : xk1;
                    A.sc[2][e] = heavy_i ? xi2 : xk2;
                    A.sc[3][e] = heavy_i ? vi0 : vk0; A.sc[4][e] = heavy_i ? vi1 : vk1;
                    A.sc[5][e] = heavy_i ? vi2 : vk2;
                    A.sc[6][e] = heavy_i ? wi - wk : wk - wi;
                    if (heavy_i) (in_i ? A.a.w : A.sc[6])[pi] = wk;
                    else (in_k ? A.b.w : A.sc[6])[pk] = wi;
                }
                (in_i ? A.a.v0 : A.sc[3])[pi] = ui0; (in_i ? A.a.v1 : A.sc[4])[pi] = ui1;
                (in_i ? A.a.v2 : A.sc[5])[pi] = ui2;
                (in_k ? A.b.v0 : A.sc[3])[pk] = uk0; (in_k ? A.b.v1 : A.sc[4])[pk] = uk1;
                (in_k ? A.b.v2 : A.sc[5])[pk] = uk2;
            }
        }
        S.performed += a;
        if (SWPM) {
            S.ca += 2 * a;
            S.na += 2 * a;
        } else if (KIND == NTC_PLAIN) {
            S.eqw += a;
        } else {
            const uint64_t am = __ballot(on_a);
            const int ne = __popcll(taken & eqm), na = __popcll(taken & ~eqm & am), nb = a - ne - na;
            S.eqw += ne;
            S.ca += na;
            S.na += na;
            S.cb += nb;
            S.nb += nb;
            if (why == MZ_WALK_LAST && single) inc ^= 1;   // the prediction for the next window
        }
        cc += a + j;
        o = D + (uint64_t)(5 * a + 3 * j);
        if (why == MZ_WALK_TRACKS) lt = min(3, lt + 1);
        else if (why == MZ_WALK_TRACK && 2 * a < T) lt = max(0, lt - 1);
        bool direct = false;
        if (why == MZ_WALK_STOP) {
            direct = ((samem >> pos) & 1) || pos == 0;   // pos 0: a pick out of range by rounding
            if ((slowm >> pos) & 1) {                     // g <= eps: two draws, no acceptance test
                direct = false;
                ++cc;
                o += 2;
            }
        }
        S.sgwm = sgwm;
        // the window's stores before the loads that follow: one wave's vector
        // memory operations stay in order, so this only holds the compiler
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        if (direct) {
            dr.seek(o);
            if (SWPM) swpm_candidate(A, c, C, S, dr, wtf, inv_w_max);
            else ntc_candidate(A, c, C, S, dr);   // Philox draws: never exhausted
            o = dr.k;
            ++cc;
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        }
    }
}

// Calls over at most NTC_WAVE_MAX_CELLS cells run every cell on a wavefront.
// Calls over more run a pass of one lane per cell, which leaves some cells to
// a second pass of one wavefront per cell.  A lane takes lane_us per candidate,
// one after another, however many cells there are (until the gathers of all
// lanes fill the memory: NTC_LANE_FILL us per candidate and cell).  The second
// pass has a latency of its own (NTC_LEFT_US), and a cell takes window_ns of the
// whole chip for its start and for each window, which reaches as far as its
// tracks do or until a particle is met again, after about sqrt(particles)
// candidates.  So each group of 64 cells picks the number of candidates up to
// which its cells run on lanes that makes the sum of its longest lane and of the
// second pass, were all groups like it, the least.
//
// us a call, all on lanes / all on wavefronts / this rule.  No particles created,
// cells of 60 particles and c candidates: 8,192 cells, c = 6 23 / 39 / 28, c = 25 75
// / 85 / 80, c = 100 276 / 246 / 234; 16,384, c = 12 45 / 84 / 50, c = 200 610 / 840
// / 624; 65,536, c = 12 127 / 278 / 135.  Splitting: 8,192, c = 100 653 / 392 / 356;
// 32,768, c = 50 631 / 720 / 564.  Cells of 2 to 125 candidates, evenly over the
// logarithm: 16,384 cells 364 / 150 / 174, splitting 911 / 394 / 415.  What the
// rule costs where lanes are right is the second launch: 9 -> 12 us for 4,097 cells
// of one candidate, 12 -> 17 us for 65,536.
#define NTC_WAVE_MAX_CELLS 4096
#define NTC_LANE_MIN 4            // candidates that always run on a lane
#define NTC_LANE_FILL 1.2e-4
#define NTC_LEFT_US 12.0
struct NtcCost {
    double lane_us, window_ns;
};
#define NTC_COST_PLAIN NtcCost{2.75, 1.8}
#define NTC_COST_SPLIT NtcCost{5.0, 2.5}
#define NTC_COST_SWPM NtcCost{5.0, 1.8}

// Whether this lane's cell (in: there is one), of n candidates among np
// particles, runs on the lane; `cells` in the call.  All 64 lanes take part.
__device__ __forceinline__ bool ntc_on_lane(bool in, int64_t n, int32_t np, int cells, const NtcCost &k) {
    const double x = in ? (double)n : 0.0, top = mz_wave_max(x);
    if (!(top > NTC_LANE_MIN)) return true;
    const double share = k.window_ns * 1e-3 * cells / __popcll(__ballot(in));
    const double wave_us = share * (1.0 + x / fmin(18.0, sqrt((double)np)));
    const double c = fmax(k.lane_us, NTC_LANE_FILL * cells);
    double best = 1e300, most = NTC_LANE_MIN;
    for (double t = NTC_LANE_MIN;; t *= 2.0) {
        const bool all = t >= top;
        const double cost = c * mz_wave_max(x <= t ? x : 0.0) +
                            (all ? 0.0 : NTC_LEFT_US + mz_wave_sum(x <= t ? 0.0 : wave_us));
        // a bound between the least and all has to be clearly better: the
        // longest lane of any group holds up the call
        if (cost < (all ? best : 0.8 * best)) {
            best = cost;
            most = t;
        }
        if (all) break;
    }
    return x <= most;
}

// Whether this lane runs its cell (in: there is one); left gets a bit for each
// cell that is left.
__device__ __forceinline__ bool ntc_stays(const NtcArgs &A, bool in, int64_t n, int32_t np, const NtcCost &k,
                                          uint64_t *left) {
    if (left) {
        const bool on = ntc_on_lane(in, n, np, A.cell_hi - A.cell_lo + 1, k);
        const uint64_t m = __ballot(!on);
        if (threadIdx.x == 0) left[blockIdx.x] = m;
        if (!on) return false;
    }
    return in;
}

// One lane per cell; cells run in parallel (64-lane workgroups, so the loop
// keeps its state in registers).  left == nullptr: every cell.
__global__ void __launch_bounds__(64) k_ntc(NtcArgs A, uint64_t *left) {
    const int c = A.cell_lo + blockIdx.x * blockDim.x + threadIdx.x;
    const bool in = c <= A.cell_hi;
    A.rp = mz_rng_resolve(A.rp);
    NtcLaneDraw dr{A.rp, mz_stream((uint64_t)c)};
    NtcCell C;
    NtcState S;
    C.n_coll = C.nla = C.nlb = 0;
    if (in) ntc_setup(A, c, dr, C, S);
    if (!ntc_stays(A, in, C.n_coll, min(C.nla, C.nlb), A.may_split ? NTC_COST_SPLIT : NTC_COST_PLAIN, left)) return;
    for (int64_t cc = 0; cc < C.n_coll; ++cc)
        if (!ntc_candidate(A, c, C, S, dr)) return;
    ntc_finish_cell(A, c, C, S);
}

// The cells left by the lanes: wavefront k of the launch looks after cells
// per k .. per k + per - 1 (per divides 64).  Up to 8,192 cells a workgroup is one
// wavefront and one cell; in larger calls, where mostly none is left, it is four,
// of several cells each, since a workgroup's start costs more than its look
// (65,536 of them 16 us).  One queue for all wavefronts costs 20 ns a cell, its
// counter's atomics one after another: 80 us for 4,096 cells.
template <class Run>
__device__ __forceinline__ void ntc_left_cells(const NtcArgs &A, const uint64_t *left, int per, Run run) {
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c0 = per * (blockIdx.x * (blockDim.x >> 6) + wv);   // from A.cell_lo
    if (A.cell_lo + c0 > A.cell_hi) return;
    uint64_t m = left[c0 >> 6] >> (c0 & 63);
    if (per < 64) m &= (1ull << per) - 1;
    for (; m; m &= m - 1) run(A.cell_lo + c0 + (int)__builtin_ctzll(m));
}

// Cell c on this wavefront (Philox draws), candidates a window at a time.
template <int KIND>
__device__ __forceinline__ void ntc_wave_cell(const NtcArgs &A, const int c) {
    NtcWaveDraw dr{A.rp, (uint64_t)c, 0, ~(uint64_t)0, 0.0, 0.0};
    NtcCell C;
    NtcState S;
    ntc_setup(A, c, dr, C, S);
    ntc_windows<KIND>(A, c, C, S, dr, 0.0, 0.0);
    if ((threadIdx.x & 63) == 0) ntc_finish_cell(A, c, C, S);
}

template <int KIND>
__global__ void __launch_bounds__(64) k_ntc_wave(NtcArgs A) {
    A.rp = mz_rng_resolve(A.rp);
    ntc_wave_cell<KIND>(A, A.cell_lo + blockIdx.x);
}

template <int KIND>
__global__ void __launch_bounds__(256) k_ntc_left(NtcArgs A, const uint64_t *left, int per) {
    A.rp = mz_rng_resolve(A.rp);
    ntc_left_cells(A, left, per, [&](int c) { ntc_wave_cell<KIND>(A, c); });
}

// Count pass of the split path: n_coll of every cell (draw 0 of its stream).
__global__ void k_ntc_count(NtcArgs A, int32_t *__restrict__ ncoll) {
    const int c = A.cell_lo + blockIdx.x * blockDim.x + threadIdx.x;
    if (c > A.cell_hi) return;
    const int32_t nla = A.a.pia.nloc[c], nlb = A.b.pia.nloc[c];
    A.rp = mz_rng_resolve(A.rp);
    MzStream st = mz_stream((uint64_t)c);
    double R = mz_rand(A.rp, st);
    double sgwm = A.sgwm[c];
    double f = floor(mz_ncoll_est(A.single, A.dt, nla, nlb, sgwm, A.V[c], R));
    if (!(f <= (double)MZ_NTC_MAX_CANDIDATES)) {
        atomicOr(&A.a.ctr->err, MZ_ERR_SCRATCH);
        f = 0.0;
    }
    ncoll[c] = (int32_t)f;
}

// Exclusive scan of n int32 values into int64 offsets (one 1024-thread block);
// total goes to *total.
__global__ void __launch_bounds__(1024) k_scan_i32(const int32_t *__restrict__ in, int64_t n,
                                                   int64_t *__restrict__ out, int64_t *__restrict__ total) {
    mz_scan_counts(in, n, out, total);
}

// Append pass: created particles of cell c go to positions
// n_total_old + coff[c] + j (1-based +1), ids from the LIFO in creation order.
__global__ void k_ntc_append(MzSpView sp, int32_t cell_lo, int32_t cell_hi, const int32_t *__restrict__ created,
                             const int64_t *__restrict__ coff, const int64_t *__restrict__ ctotal,
                             const int64_t *__restrict__ soff, const double *const *sc, int64_t sc_off,
                             MzCounters snap) {
    const int c = cell_lo + blockIdx.x;
    if (c > cell_hi) return;
    const int32_t k = created[c];
    if (k == 0) return;
    const int64_t base = (int64_t)snap.n_total + coff[c];  // 0-based first new slot
    for (int j = threadIdx.x; j < k; j += blockDim.x) {
        int64_t dst = base + j;
        if (dst >= sp.cap) {
            atomicOr(&sp.ctr->err, MZ_ERR_CAPACITY);
            continue;
        }
        int64_t src = sc_off + soff[c] + j;
        sp.x0[dst] = sc[0][src]; sp.x1[dst] = sc[1][src]; sp.x2[dst] = sc[2][src];
        sp.v0[dst] = sc[3][src]; sp.v1[dst] = sc[4][src]; sp.v2[dst] = sc[5][src];
        sp.w[dst] = sc[6][src];
        int64_t q = coff[c] + j;   // global creation number
        int32_t idv = q < snap.nbuffer ? sp.buffer[snap.nbuffer - 1 - q]
                                       : (int32_t)(snap.length + 1 + (q - snap.nbuffer));
        sp.id[dst] = idv;
        sp.key[dst] = c + 1;
    }
    if (threadIdx.x == 0) {
        // update_particle_indexer_new_particle! applied k times
        sp.pia.nloc[c] += k;
        sp.pia.n2[c] += k;
        if (sp.pia.start2[c] <= 0) sp.pia.start2[c] = (int32_t)(base + 1);
        sp.pia.end2[c] = (int32_t)(base + k);
    }
    (void)ctotal;
}

// Counters after the append: n_total, n_pos, and the LIFO / length as a run of
// resize! + pops leaves them.
__global__ void k_ntc_finish(MzSpView sp, const int64_t *__restrict__ ctotal, MzCounters snap) {
    const int64_t tot = *ctotal;
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        sp.ctr->created = (int32_t)tot;
        if (tot == 0) return;
        int64_t nt = (int64_t)snap.n_total + tot;
        if (nt > sp.cap) {
            atomicOr(&sp.ctr->err, MZ_ERR_CAPACITY);
            nt = sp.cap;
        }
        sp.ctr->n_total = (int32_t)nt;
        sp.ctr->n_pos = max(snap.n_pos, sp.ctr->n_total);
        if (tot <= snap.nbuffer) {
            sp.ctr->nbuffer = snap.nbuffer - (int32_t)tot;
        } else {
            int64_t R = tot - snap.nbuffer;
            int64_t chunks = (R + MZ_DELTA_PARTICLES - 1) / MZ_DELTA_PARTICLES;
            int64_t L2 = snap.length + chunks * MZ_DELTA_PARTICLES;
            sp.ctr->length = (int32_t)L2;
            sp.ctr->nbuffer = (int32_t)(L2 - snap.length - R);
        }
    }
    // the remaining free ids after a resize: buffer[0..nbuffer) = L', L'-1, ...
    if (tot > snap.nbuffer) {
        int64_t R = tot - snap.nbuffer;
        int64_t chunks = (R + MZ_DELTA_PARTICLES - 1) / MZ_DELTA_PARTICLES;
        int64_t L2 = snap.length + chunks * MZ_DELTA_PARTICLES;
        int64_t nbuf = L2 - snap.length - R;
        if (nbuf > sp.bufcap) {
            if (threadIdx.x == 0) atomicOr(&sp.ctr->err, MZ_ERR_BUFFER);
            return;
        }
        for (int64_t i = threadIdx.x; i < nbuf; i += blockDim.x) sp.buffer[i] = (int32_t)(L2 - i);
    }
}

static NtcArgs base_args(mz_store *h, int s1, int s2, double dt, const double *dV, double dw_tol, int equal_weight,
                         uint64_t tag, int rng_mode, int cell_lo, int cell_hi) {
    NtcArgs A{};
    A.a = mz_view(h->sp[s1 - 1]);
    A.b = mz_view(h->sp[s2 - 1]);
    A.single = s1 == s2;
    A.equal_weight = equal_weight;
    A.cell_lo = cell_lo - 1;
    A.cell_hi = cell_hi - 1;
    A.dt = dt;
    A.dw_tol = dw_tol;
    const MzInteraction &it = h->inter[(s1 - 1) * h->n_species + (s2 - 1)];
    A.mu1 = it.mu1; A.mu2 = it.mu2; A.factor = it.factor; A.expo = it.expo;
    A.V = dV;
    size_t pair = (size_t)(s1 - 1) * h->n_species + (s2 - 1);
    A.sgwm = h->d_sgwm + pair * h->n_cells;
    A.cnt = h->d_cfcnt + pair * h->n_cells * 5;
    A.rp = mz_rng_params(h, 0, tag, rng_mode);
    return A;
}

// the launch shape of ntc_left_cells
struct NtcLeftShape {
    dim3 grid, block;
    int per;
};
static NtcLeftShape ntc_left_shape(int ncells) {
    const int waves = ncells <= 8192 ? 1 : 4;
    int per = 1;
    while (per < 64 && ncells > 16384 * per) per *= 2;
    return NtcLeftShape{dim3((ncells + waves * per - 1) / (waves * per)), dim3(64 * waves), per};
}

// The candidate loops over ncells cells; replayed draws run one lane per cell.
static void launch_k_ntc(mz_store *h, const NtcArgs &A, int ncells) {
    const dim3 lanes((ncells + 63) / 64);
    uint64_t *const left = h->d_ntc_left;
    if (A.rp.mode != 0) {
        hipLaunchKernelGGL(k_ntc, lanes, dim3(64), 0, h->stream, A, (uint64_t *)nullptr);
    } else if (ncells <= NTC_WAVE_MAX_CELLS) {
        hipLaunchKernelGGL(A.may_split ? k_ntc_wave<NTC_SPLIT> : k_ntc_wave<NTC_PLAIN>, dim3(ncells), dim3(64), 0,
                           h->stream, A);
    } else {
        hipLaunchKernelGGL(k_ntc, lanes, dim3(64), 0, h->stream, A, left);
        const NtcLeftShape ls = ntc_left_shape(ncells);
        hipLaunchKernelGGL(A.may_split ? k_ntc_left<NTC_SPLIT> : k_ntc_left<NTC_PLAIN>, ls.grid, ls.block, 0, h->stream,
                           A, (const uint64_t *)left, ls.per);
    }
}

int mz_launch_ntc_equal(mz_store *h, int s1, int s2, double dt, const double *dV, double dw_tol, int equal_weight,
                        uint64_t tag, int rng_mode, int cell_lo, int cell_hi, const uint64_t *step_ptr) {
    NtcArgs A = base_args(h, s1, s2, dt, dV, dw_tol, equal_weight, tag, rng_mode, cell_lo, cell_hi);
    A.may_split = 0;
    A.rp.step_ptr = step_ptr;
    A.rp.phase = 1;
    int ncells = cell_hi - cell_lo + 1;
    launch_k_ntc(h, A, ncells);
    MZ_HIP(hipGetLastError());
    return 0;
}

static int launch_ntc_split(mz_store *h, int s1, int s2, double dt, const double *dV, double dw_tol, uint64_t tag,
                            int rng_mode, int cell_lo, int cell_hi) {
    NtcArgs A = base_args(h, s1, s2, dt, dV, dw_tol, 0, tag, rng_mode, cell_lo, cell_hi);
    A.may_split = 1;
    const int nc = h->n_cells;
    const int ncells = cell_hi - cell_lo + 1;
    int32_t *ncoll = (int32_t *)mz_scratch(h, "ntc_ncoll", (size_t)nc * sizeof(int32_t));
    int64_t *soff = (int64_t *)mz_scratch(h, "ntc_soff", (size_t)(nc + 1) * sizeof(int64_t));
    int32_t *created = (int32_t *)mz_scratch(h, "ntc_created", (size_t)2 * nc * sizeof(int32_t));
    int64_t *coff = (int64_t *)mz_scratch(h, "ntc_coff", (size_t)2 * (nc + 1) * sizeof(int64_t));
    MZ_CHECK(ncoll && soff && created && coff, "ntc: scratch allocation failed");
    MZ_HIP(hipMemsetAsync(ncoll, 0, (size_t)nc * sizeof(int32_t), h->stream));
    MZ_HIP(hipMemsetAsync(created, 0, (size_t)2 * nc * sizeof(int32_t), h->stream));
    hipLaunchKernelGGL(k_ntc_count, dim3((ncells + 255) / 256), dim3(256), 0, h->stream, A, ncoll);
    hipLaunchKernelGGL(k_scan_i32, dim3(1), dim3(1024), 0, h->stream, ncoll, (int64_t)nc, soff, soff + nc);
    int64_t total = 0;
    MZ_HIP(hipMemcpyAsync(&total, soff + nc, sizeof(int64_t), hipMemcpyDeviceToHost, h->stream));
    MZ_HIP(hipStreamSynchronize(h->stream));
    int64_t cap = std::max<int64_t>(total, 1);
    double *sc = (double *)mz_scratch(h, "ntc_sc", (size_t)7 * 2 * cap * sizeof(double));
    MZ_CHECK(sc != nullptr, "ntc: creation scratch allocation failed");
    for (int f = 0; f < 7; ++f) A.sc[f] = sc + (size_t)f * 2 * cap;
    A.sc_cap = cap;
    A.ncoll_in = ncoll;
    A.soff = soff;
    // created is indexed [species half][cell]; the kernel writes half 1 at cell_hi + 1 + c
    A.created = created;
    launch_k_ntc(h, A, ncells);
    MZ_HIP(hipGetLastError());
    // append per species half
    double **scp = (double **)mz_scratch(h, "ntc_scp", 7 * sizeof(double *));
    MZ_CHECK(scp != nullptr, "ntc: scratch allocation failed");
    MZ_HIP(hipMemcpy(scp, A.sc, 7 * sizeof(double *), hipMemcpyHostToDevice));
    for (int half = 0; half < (A.single ? 1 : 2); ++half) {
        int sidx = half == 0 ? s1 : s2;
        const int32_t *cr = created + (half == 0 ? 0 : (int64_t)(A.cell_hi + 1));
        int64_t *co = coff + (size_t)half * (nc + 1);
        MzCounters snap;
        int r = mz_read_counters(h, sidx, &snap);
        if (r) return r;
        // created[] for half 1 is offset by cell_hi + 1 entries; scan the used range
        hipLaunchKernelGGL(k_scan_i32, dim3(1), dim3(1024), 0, h->stream, cr, (int64_t)(A.cell_hi + 1), co,
                           co + nc);
        hipLaunchKernelGGL(k_ntc_append, dim3(ncells), dim3(64), 0, h->stream, mz_view(h->sp[sidx - 1]), A.cell_lo,
                           A.cell_hi, cr, co, co + nc, soff, (const double *const *)scp, (int64_t)half * cap, snap);
        hipLaunchKernelGGL(k_ntc_finish, dim3(1), dim3(256), 0, h->stream, mz_view(h->sp[sidx - 1]), co + nc, snap);
        MZ_HIP(hipGetLastError());
    }
    return 0;
}

// The cell volumes V[n_cells] of an NTC or SWPM call on the device.  They upload
// only when they differ from the last upload; an upload first waits for the
// store's stream, whose queued kernels may still read the previous values.
static int upload_ntc_volumes(mz_store *h, const double *V, const double **out) {
    double *v = (double *)mz_scratch(h, "ntc_V", h->n_cells * sizeof(double));
    MZ_CHECK(v != nullptr, "ntc: scratch allocation failed");
    if (h->ntc_V_up.size() != (size_t)h->n_cells ||
        std::memcmp(h->ntc_V_up.data(), V, h->n_cells * sizeof(double)) != 0 || h->ntc_V_dev != v) {
        MZ_HIP(hipStreamSynchronize(h->stream));
        MZ_HIP(hipMemcpy(v, V, h->n_cells * sizeof(double), hipMemcpyHostToDevice));
        h->ntc_V_up.assign(V, V + h->n_cells);
        h->ntc_V_dev = v;
    }
    *out = v;
    return 0;
}

extern "C" int mz_ntc(mz_store *h, int32_t s1, int32_t s2, double dt, const double *V, double dw_tol,
                      int32_t equal_weight, uint64_t tag, int32_t rng_mode, int32_t cell_lo, int32_t cell_hi) {
    MZ_CHECK(s1 >= 1 && s1 <= h->n_species && s2 >= 1 && s2 <= h->n_species, "ntc: bad species");
    MZ_CHECK(cell_lo >= 1 && cell_hi <= h->n_cells && cell_lo <= cell_hi, "ntc: bad cell range");
    MZ_CHECK(h->inter[(s1 - 1) * h->n_species + (s2 - 1)].set, "ntc: interaction not set");
    MZ_CHECK(rng_mode == 0 || (rng_mode == 1 && h->d_replay[0]), "ntc: replay table not set");
    const double *dV = h->d_V;
    if (V) {
        int r = upload_ntc_volumes(h, V, &dV);
        if (r) return r;
    } else {
        MZ_CHECK(h->has_grid, "ntc: V is NULL and no grid is set");
    }
    MzTimed tm(h, "ntc");
    if (equal_weight) return mz_launch_ntc_equal(h, s1, s2, dt, dV, dw_tol, 1, tag, rng_mode, cell_lo, cell_hi);
    return launch_ntc_split(h, s1, s2, dt, dV, dw_tol, tag, rng_mode, cell_lo, cell_hi);
}

// The reference's loop of per-cell ntc! calls (test/test_1D_couette.jl:67-71)
// as one call: cell cells[k] with volume V[k], in list order.  A maximal run
// of consecutive ascending cells launches as one range (its cells are
// independent and its splits append in cell order), runs launch one after
// another, so the result is the sequential loop's for any list.
extern "C" int mz_ntc_cells(mz_store *h, int32_t s1, int32_t s2, double dt, const int32_t *cells, const double *V,
                            int32_t n, double dw_tol, int32_t equal_weight, uint64_t tag, int32_t rng_mode) {
    MZ_CHECK(s1 >= 1 && s1 <= h->n_species && s2 >= 1 && s2 <= h->n_species, "ntc_cells: bad species");
    MZ_CHECK(h->inter[(s1 - 1) * h->n_species + (s2 - 1)].set, "ntc_cells: interaction not set");
    MZ_CHECK(rng_mode == 0 || (rng_mode == 1 && h->d_replay[0]), "ntc_cells: replay table not set");
    MZ_CHECK(n >= 0 && (n == 0 || (cells != nullptr && V != nullptr)), "ntc_cells: bad cell list");
    for (int32_t k = 0; k < n; ++k) MZ_CHECK(cells[k] >= 1 && cells[k] <= h->n_cells, "ntc_cells: cell out of range");
    if (n == 0) return 0;
    std::vector<double> full = h->ntc_V_up.size() == (size_t)h->n_cells ? h->ntc_V_up
                                                                           : std::vector<double>(h->n_cells, 1.0);
    MzTimed tm(h, "ntc");
    int32_t k0 = 0;
    while (k0 < n) {
        int32_t k1 = k0 + 1;
        while (k1 < n && cells[k1] == cells[k1 - 1] + 1) ++k1;
        for (int32_t k = k0; k < k1; ++k) full[cells[k] - 1] = V[k];
        const double *dv = nullptr;
        int r = upload_ntc_volumes(h, full.data(), &dv);
        if (r) return r;
        const int32_t lo = cells[k0], hi = cells[k1 - 1];
        r = equal_weight ? mz_launch_ntc_equal(h, s1, s2, dt, dv, dw_tol, 1, tag, rng_mode, lo, hi)
                         : launch_ntc_split(h, s1, s2, dt, dv, dw_tol, tag, rng_mode, lo, hi);
        if (r) return r;
        k0 = k1;
    }
    return 0;
}

// ===========================================================================
// swpm! (collision_swpm.jl:201-288): single-species collisions of
// variable-weight particles.  A cell's loop is sequential (the running
// (sigma g)_max, and particles created by the loop are candidates of the same
// loop) and runs as NTC's do: in windows of a wavefront, or on a lane.  An accepted pair gives up
// min(w_i, w_k) / (1 + G) of each weight to two new particles at the pair's
// positions, which then take the pair's post-collision velocities
// (scatter_vhs!); the pair keeps its velocities.  Created particles go to
// per-cell scratch and are appended in cell order as for NTC splits.  For
// this method the pair's (sigma g w)_max array holds (sigma g)_max.

// Count pass: w_max of every cell, its candidate count (draw 0 of its
// stream, compute_n_coll_single_species, collision_swpm.jl:171-174) and the
// scratch it may need (two particles per candidate); one wave per cell.
__global__ void __launch_bounds__(256) k_swpm_count(NtcArgs A, double G, int32_t *__restrict__ ncoll,
                                                    int32_t *__restrict__ ssz, double *__restrict__ wmax) {
    const int c = A.cell_lo + blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (c > A.cell_hi) return;
    const int32_t n1 = A.a.pia.n1[c], n2 = A.a.pia.n2[c] > 0 ? A.a.pia.n2[c] : 0, np = A.a.pia.nloc[c];
    double w_max = 0.0;
    for (int32_t li = lane; li < n1 + n2; li += 64) {
        const double w = A.a.w[slot_of(A.a, c, li, n1, n2)];
        w_max = w > w_max ? w : w_max;
    }
    w_max = mz_wave_max(w_max);
    if (lane != 0) return;
    A.rp = mz_rng_resolve(A.rp);
    MzStream st = mz_stream((uint64_t)c);
    const double R = mz_rand(A.rp, st);
    double f = floor(0.5 * A.dt * (double)np * (double)(np - 1) * A.sgwm[c] * w_max * (G + 1) / A.V[c] + R);
    if (!(f <= (double)MZ_NTC_MAX_CANDIDATES / 2)) {   // also catches NaN estimates
        atomicOr(&A.a.ctr->err, MZ_ERR_SCRATCH);
        f = 0.0;
    }
    ncoll[c] = (int32_t)f;
    ssz[c] = 2 * (int32_t)f;
    wmax[c] = w_max;
}

__device__ __forceinline__ void swpm_setup(const NtcArgs &A, const int c, NtcCell &C, NtcState &S) {
    C.n1a = C.n1b = A.a.pia.n1[c];
    C.n2a = C.n2b = A.a.pia.n2[c] > 0 ? A.a.pia.n2[c] : 0;
    C.nla = C.nlb = A.a.pia.nloc[c];
    C.n_coll = A.ncoll_in[c];
    C.s_base = A.soff[c];
    S.na = S.nb = C.nla;
    S.ca = S.cb = 0;
    S.performed = S.eqw = 0;
    S.sgwm = A.sgwm[c];
}

__device__ __forceinline__ void swpm_finish(const NtcArgs &A, const int c, const NtcCell &C, const NtcState &S) {
    A.sgwm[c] = S.sgwm;
    int32_t *cn = A.cnt + (int64_t)c * 5;
    cn[0] = C.nla;
    cn[1] = C.nla;
    cn[2] = (int32_t)C.n_coll;
    cn[3] = S.performed;
    cn[4] = 0;
    A.created[c] = S.ca;
}

// One lane per cell (k_ntc's rule).
__global__ void __launch_bounds__(64) k_swpm(NtcArgs A, double G, const double *__restrict__ wmax, uint64_t *left) {
    const int c = A.cell_lo + blockIdx.x * blockDim.x + threadIdx.x;
    const bool in = c <= A.cell_hi;
    if (!ntc_stays(A, in, in ? A.ncoll_in[c] : 0, in ? A.a.pia.nloc[c] : 0, NTC_COST_SWPM, left)) return;
    A.rp = mz_rng_resolve(A.rp);
    NtcLaneDraw dr{A.rp, mz_stream((uint64_t)c)};
    dr.seek(1);
    NtcCell C;
    NtcState S;
    swpm_setup(A, c, C, S);
    const double wtf = 1.0 / (1.0 + G), inv_w_max = 1.0 / wmax[c];
    for (int64_t cc = 0; cc < C.n_coll; ++cc)
        if (!swpm_candidate(A, c, C, S, dr, wtf, inv_w_max)) return;
    swpm_finish(A, c, C, S);
}

// Cell c on this wavefront (Philox draws), candidates a window at a time.
__device__ __forceinline__ void swpm_wave_cell(const NtcArgs &A, const int c, double G, const double *wmax) {
    NtcWaveDraw dr{A.rp, (uint64_t)c, 1, ~(uint64_t)0, 0.0, 0.0};
    NtcCell C;
    NtcState S;
    swpm_setup(A, c, C, S);
    ntc_windows<NTC_SWPM>(A, c, C, S, dr, 1.0 / (1.0 + G), 1.0 / wmax[c]);
    if ((threadIdx.x & 63) == 0) swpm_finish(A, c, C, S);
}

__global__ void __launch_bounds__(64) k_swpm_wave(NtcArgs A, double G, const double *__restrict__ wmax) {
    A.rp = mz_rng_resolve(A.rp);
    swpm_wave_cell(A, A.cell_lo + blockIdx.x, G, wmax);
}

__global__ void __launch_bounds__(256) k_swpm_left(NtcArgs A, double G, const double *__restrict__ wmax,
                                                   const uint64_t *left, int per) {
    A.rp = mz_rng_resolve(A.rp);
    ntc_left_cells(A, left, per, [&](int c) { swpm_wave_cell(A, c, G, wmax); });
}

extern "C" int mz_swpm(mz_store *h, int32_t species, double G, double dt, const double *V, uint64_t tag,
                       int32_t rng_mode, int32_t cell_lo, int32_t cell_hi) {
    MZ_CHECK(species >= 1 && species <= h->n_species, "swpm: bad species");
    MZ_CHECK(cell_lo >= 1 && cell_hi <= h->n_cells && cell_lo <= cell_hi, "swpm: bad cell range");
    MZ_CHECK(G >= 0.0, "swpm: G must be non-negative");
    MZ_CHECK(h->inter[(species - 1) * h->n_species + (species - 1)].set, "swpm: interaction not set");
    MZ_CHECK(rng_mode == 0 || (rng_mode == 1 && h->d_replay[0]), "swpm: replay table not set");
    const double *dV = h->d_V;
    if (V) {
        int r = upload_ntc_volumes(h, V, &dV);
        if (r) return r;
    } else {
        MZ_CHECK(h->has_grid, "swpm: V is NULL and no grid is set");
    }
    NtcArgs A = base_args(h, species, species, dt, dV, 0.0, 0, tag, rng_mode, cell_lo, cell_hi);
    A.may_split = 1;
    const int nc = h->n_cells;
    const int ncells = cell_hi - cell_lo + 1;
    int32_t *ncoll = (int32_t *)mz_scratch(h, "ntc_ncoll", (size_t)nc * sizeof(int32_t));
    int32_t *ssz = (int32_t *)mz_scratch(h, "swpm_ssz", (size_t)nc * sizeof(int32_t));
    double *wmax = (double *)mz_scratch(h, "swpm_wmax", (size_t)nc * sizeof(double));
    int64_t *soff = (int64_t *)mz_scratch(h, "ntc_soff", (size_t)(nc + 1) * sizeof(int64_t));
    int32_t *created = (int32_t *)mz_scratch(h, "ntc_created", (size_t)2 * nc * sizeof(int32_t));
    int64_t *coff = (int64_t *)mz_scratch(h, "ntc_coff", (size_t)2 * (nc + 1) * sizeof(int64_t));
    MZ_CHECK(ncoll && ssz && wmax && soff && created && coff, "swpm: scratch allocation failed");
    MZ_HIP(hipMemsetAsync(ncoll, 0, (size_t)nc * sizeof(int32_t), h->stream));
    MZ_HIP(hipMemsetAsync(ssz, 0, (size_t)nc * sizeof(int32_t), h->stream));
    MZ_HIP(hipMemsetAsync(created, 0, (size_t)2 * nc * sizeof(int32_t), h->stream));
    {
        MzTimed tm(h, "swpm");
        hipLaunchKernelGGL(k_swpm_count, dim3((ncells + 3) / 4), dim3(256), 0, h->stream, A, G, ncoll, ssz, wmax);
        hipLaunchKernelGGL(k_scan_i32, dim3(1), dim3(1024), 0, h->stream, ssz, (int64_t)nc, soff, soff + nc);
        int64_t total = 0;
        MZ_HIP(hipMemcpyAsync(&total, soff + nc, sizeof(int64_t), hipMemcpyDeviceToHost, h->stream));
        MZ_HIP(hipStreamSynchronize(h->stream));
        const int64_t cap = std::max<int64_t>(total, 1);
        double *sc = (double *)mz_scratch(h, "ntc_sc", (size_t)7 * cap * sizeof(double));
        MZ_CHECK(sc != nullptr, "swpm: creation scratch allocation failed");
        for (int f = 0; f < 7; ++f) A.sc[f] = sc + (size_t)f * cap;
        A.sc_cap = cap;
        A.ncoll_in = ncoll;
        A.soff = soff;
        A.created = created;
        // the rule of launch_k_ntc
        const double *const wm = wmax;
        const dim3 lanes((ncells + 63) / 64);
        uint64_t *const left = h->d_ntc_left;
        if (rng_mode != 0) {
            hipLaunchKernelGGL(k_swpm, lanes, dim3(64), 0, h->stream, A, G, wm, (uint64_t *)nullptr);
        } else if (ncells <= NTC_WAVE_MAX_CELLS) {
            hipLaunchKernelGGL(k_swpm_wave, dim3(ncells), dim3(64), 0, h->stream, A, G, wm);
        } else {
            hipLaunchKernelGGL(k_swpm, lanes, dim3(64), 0, h->stream, A, G, wm, left);
            const NtcLeftShape ls = ntc_left_shape(ncells);
            hipLaunchKernelGGL(k_swpm_left, ls.grid, ls.block, 0, h->stream, A, G, wm, (const uint64_t *)left, ls.per);
        }
        MZ_HIP(hipGetLastError());
        double **scp = (double **)mz_scratch(h, "ntc_scp", 7 * sizeof(double *));
        MZ_CHECK(scp != nullptr, "swpm: scratch allocation failed");
        MZ_HIP(hipMemcpy(scp, A.sc, 7 * sizeof(double *), hipMemcpyHostToDevice));
        MzCounters snap;
        int r = mz_read_counters(h, species, &snap);
        if (r) return r;
        hipLaunchKernelGGL(k_scan_i32, dim3(1), dim3(1024), 0, h->stream, created, (int64_t)(A.cell_hi + 1), coff,
                           coff + nc);
        hipLaunchKernelGGL(k_ntc_append, dim3(ncells), dim3(64), 0, h->stream, mz_view(h->sp[species - 1]), A.cell_lo,
                           A.cell_hi, created, coff, coff + nc, soff, (const double *const *)scp, (int64_t)0, snap);
        hipLaunchKernelGGL(k_ntc_finish, dim3(1), dim3(256), 0, h->stream, mz_view(h->sp[species - 1]), coff + nc, snap);
    }
    MZ_HIP(hipGetLastError());
    return 0;
}
