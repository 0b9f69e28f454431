// The slice-run walk: the charged segments of traverse.h's step walk, gathered piece by piece with the lane's
// slice carried along instead of derived anew in every step.
//
// The lanes of a wave (64 detector rows of one column) share the xy pieces of every plane step; they differ in z
// only, and a lane changes slice rarely (the cone's slopes: every 20 to 60 steps on a 0.5 mm / 1 mm grid).  So the
// walk keeps, per lane, the slice it is in and the position of its next slice plane, and takes the xy pieces
// of up to `nb` steps at a time, few enough that no lane meets two slice planes in them:
//  - the lanes that meet a plane in the block find the piece that holds it, and gather its two parts for themselves;
//  - main loop: every piece before that one goes to the lane's slice, those after it to the next one.  Column and
//    length come from the wave's LDS table (one 16-byte broadcast read), so a piece takes nine vector instructions (two
//    compares and selects against the uniform piece number, one address, two for the length, two multiply-adds for
//    two channels), against ~90 when each step formed its own slice indices and crossings;
//  - the parts are charged, all lanes of the block together.
// Nothing is read of a voxel that the lane does not charge: the piece that holds the plane, and the places past the end of a
// batch of gathers, are read off the volume (zeros), as a length of 0 would make a NaN of an infinite voxel.
// The reference's rules hold as in the step walk: midpoint truncation (slice 0 takes the truncated (-1, 0) range
// too), the z = 0 plane splits nothing (the whole piece goes to its midpoint's slice), the inscribed-circle test at
// the midpoint, and equal crossing distances charge the whole chord once.  Where those need a part's own midpoint
// (a step at the circle's boundary, equal distances, a plane grid off the voxel grid) the parts are formed as the
// step walk forms its segments.
// What bounds it: on the 512x512x128 / 360-angle projection the gathers' traffic beyond L2 (7.6e10 bytes at 7.3 TB/s);
// the step walk took 20.7 ms there, bound by vector issue (1.19e10 wave-instructions, now 4.6e9), this walk 10.45 ms.
// A piece's length is its extent along the major axis times the ray's length factor, formed in FP64 and rounded once per
// piece as the step walk does.  Extent and factor rounded to FP32 first would shift a whole ray by up to 6e-8; the full scan
// takes the same time either way, 320x320x77 at 0.977 mm / 120 angles 1.87 against 1.80 ms, six u16 maps 1.47 against
// 1.50.  FP32 sums of equal terms (a constant map) round one way, and by the terms' own digits, so lengths scaled once at
// the end would leave a log projection 1e-7 off the step walk's there.
#pragma once

#include "traverse.h"

namespace vcbct {

// One xy piece: its extent along the major axis and its voxel column.
struct PieceRec {
    double len;
    int cb, pad;
};

// One step: the positions of its end plane and minor crossing relative to the source (as StepRec), and in flags
// STEP_SPLITV, STEP_OK0 / STEP_OK1 (the piece is in the list), RUN_SPECIAL, and the list position of its first
// piece from bit RUN_SHIFT on.
struct RunStep {
    double dk, dv;
    int flags;
};
enum { RUN_SPECIAL = 32, RUN_SHIFT = 8 };

struct RunLds {
    double dk[64], dv[64];
    int flags[64];
    PieceRec pieces[128];
};

typedef PieceRec OrderedPiece;  // (the ordered walk's)
struct OrderedLds {
    WaveLds table;
    OrderedPiece pieces[128];
};

// Scratch of one wave for any of the walks.
union WalkLds {
    WaveLds table;
    RunLds runs;
    OrderedLds ordered;
};

// Step k's record and its pieces (has0 / has1: charged by lanes that are in range).  Returns whether the
// reference's loop reaches the step.
template <bool ALIGNED>
__host__ __device__ __forceinline__ bool make_run_step(const ProjGeom& g, const RayCtx& r, const ChargeC& c, int k,
                                                       RunStep& t, PieceRec& p0, PieceRec& p1, bool& has0,
                                                       bool& has1) {
#pragma clang fp contract(fast)
    const double up = plane_u(r, k - 1, g.s);
    const double uk = plane_u(r, k, g.s);
    const double vp = (up - r.su) * r.dv + r.sv;
    const double dup = up - r.su, duk = uk - r.su;
    const double vk = duk * r.dv + r.sv;
    const bool inprev = up <= g.lim_u && up >= -g.lim_u && vp <= g.lim_u && vp >= -g.lim_u;
    const int vma = (int)(vk * g.inv_s);
    const int vmap = (int)(vp * g.inv_s);
    const bool hv = r.vmove && ((vma != vmap) || !(vk * vp > 0.0));
    double uv = uk;
    if (hv) {
        const double vb = (vma * g.s) - ((vk <= 0 && r.dirv < 0) || (vk >= 0 && r.dirv > 0) ? 0.0 : r.dirv * g.s);
        uv = (vb - r.sv) * r.duv + r.su;
    }
    const bool splitv = hv && fabs(uk - uv) != 0.0;
    const double a1 = splitv ? uv : uk;
    const double dv = uv - r.su, d1 = a1 - r.su;
    const double vv = dv * r.dv + r.sv;  // v at the minor crossing
    const double va1 = splitv ? vv : vk;
    const double m0 = (dup + d1) * 0.5, m1 = (dv + duk) * 0.5;
    const double vm0 = m0 * r.dv + r.sv, vm1 = m1 * r.dv + r.sv;
    const int imin0 = (int)(vm0 * c.smin + c.nmaj);
    const int imin1 = (int)(vm1 * c.smin + c.nmaj);
    int imaj0, imaj1;
    if (ALIGNED) {
        imaj0 = imaj1 = (int)((up + uk) * 0.5 * c.smaj + c.nmaj);
    } else {
        imaj0 = major_index(g, r, c, up, a1);
        imaj1 = major_index(g, r, c, uv, uk);
    }
    const double um0 = m0 + r.su, um1 = m1 + r.su;
    has0 = (unsigned)imaj0 < (unsigned)g.N && (unsigned)imin0 < (unsigned)g.N && um0 * um0 + vm0 * vm0 < c.rmax2;
    has1 = splitv && (unsigned)imaj1 < (unsigned)g.N && (unsigned)imin1 < (unsigned)g.N &&
           um1 * um1 + vm1 * vm1 < c.rmax2;
    // the circle's boundary crosses the chord (margins as in make_step): sub-pieces are tested one by one
    double lo, hi;
    chord_r2(up, vp, uk, vk, lo, hi);
    const bool circ = hi >= c.rmax2 - 1e-9 && lo <= c.rmax2 + 1e-9;
    t.dk = duk;
    t.dv = dv;
    p0.cb = (int)((unsigned)imin0 * (unsigned)c.mstride + (unsigned)imaj0 * (unsigned)c.majmul);
    p1.cb = (int)((unsigned)imin1 * (unsigned)c.mstride + (unsigned)imaj1 * (unsigned)c.majmul);
    p0.len = fabs(d1 - dup);
    p1.len = fabs(duk - dv);
    t.flags = (splitv ? STEP_SPLITV : 0) | (has0 ? STEP_OK0 : 0) | (has1 ? STEP_OK1 : 0) |
              (circ || !ALIGNED ? RUN_SPECIAL : 0);
    return inprev;
}

// |dz/du| of a ray, rounded up.
__host__ __device__ __forceinline__ float run_slope(const RayCtx& r) { return (float)fabs(r.dz) * 1.000001f; }

// The largest number of steps a block may take so that no lane meets two slice planes in it: `slope` the
// largest |dz/du| of the wave's lanes.  0: two planes can fall into one step (the step walk takes those).
__host__ __device__ __forceinline__ int run_block_steps(const ProjGeom& g, float slope) {
    const double n = g.t / ((double)slope * g.s) * (1.0 - 1e-6);
    return n >= 64.0 ? 64 : (n >= 1.0 ? (int)n : 0);
}

// Pieces [pa, pb) of the list: before first_new from slice offset zo, from gap_end on from zn, none between.  By the
// accumulator's own form, or in two passes.
template <class Acc>
__host__ __device__ __forceinline__ auto run_gaps(Acc& acc, const PieceRec* p, int pa, int pb, int first_new,
                                                  int gap_end, int zo, int zn, double K, int)
    -> decltype(acc.run_gaps(p, pa, pb, first_new, gap_end, zo, zn, K)) {
    acc.run_gaps(p, pa, pb, first_new, gap_end, zo, zn, K);
}
template <class Acc>
__host__ __device__ __forceinline__ void run_gaps(Acc& acc, const PieceRec* p, int pa, int pb, int first_new,
                                                  int gap_end, int zo, int zn, double K, long) {
    acc.run(p, pa, pb, INT_MAX, first_new, 0.0f, zo, (int)Acc::kOut, K);
    acc.run(p, pa, pb, INT_MAX, gap_end, 0.0f, (int)Acc::kOut, zn, K);
}

// Walks plane steps [kmin, kmax] of one wave (lanes with a common xy path, `nb` from run_block_steps).
// Acc: float accumulator with load(cell, q) (cell outside the volume: zeros), add(q, length), run_gaps() or run() for a
// list of pieces, a record type Q, and kOut, a cell offset that no column brings back into the volume.
template <bool ALIGNED, class Acc>
__host__ __device__ __forceinline__ void walk_runs(const ProjGeom& g, const RayCtx& r_in, bool active, int kmin,
                                                   int kmax, int nb, Acc& acc, RunLds* lds) {
#pragma clang fp contract(fast)
#ifdef __HIP_DEVICE_COMPILE__
    RayCtx r = r_in;  // the shared xy path from the first lane (scalar registers), as in traverse_table
    r.ui = first_lane(r_in.ui);
    r.uf = first_lane(r_in.uf);
    r.vi = first_lane(r_in.vi);
    r.vf = first_lane(r_in.vf);
    r.uin = first_lane(r_in.uin);
    r.pha = first_lane(r_in.pha);
    r.dirv = first_lane(r_in.dirv);
    const int lane = threadIdx.x & 63;
#else
    const RayCtx& r = r_in;
#endif
    constexpr bool kEarly = sizeof(typename Acc::Q) <= (ALIGNED ? 8 : 12);
    const bool on = active && r.hit;
    const ChargeC c = charge_consts(g, r);
    const double u0 = r.uin;
    const double v0 = (u0 - r.su) * r.dv + r.sv;
    if (!(u0 <= g.lim_u && u0 >= -g.lim_u && v0 <= g.lim_u && v0 >= -g.lim_u)) return;
    int k = kmin;
    if (k <= 1) {  // the lumped entry segment
        const Seg sg = make_seg<false, false>(g, r, c, r.ui, u0, on, 0, false);
        typename Acc::Q q;
        acc.load(sg.ok ? sg.cell : Acc::kOut, q);
        acc.add(q, sg.ok ? (float)sg.rr : 0.0f);
        k = 1;
    }
    // The slice index along the walk is fA D + fB, D the position in walking direction.  The lane's logical slice
    // (slice -1: the truncated range, charged to slice 0) and its next plane, f = il + up.
    const double fA = r.pha * r.dz * c.ninv_t;
    const double duzD = r.pha * r.duz;
    const int up = fA > 0.0 ? 1 : 0, sgn = fA > 0.0 ? 1 : -1;
    double D0 = (plane_u(r, k - 1, g.s) - r.su) * r.pha;  // the plane before the first step
    const int nzm = (int)c.nzm;
    // the position of plane f = mm, z = (nzm - mm) t, in the step walk's expression (a plane met on the way to z = 0
    // is formed from the one after it, as the reference forms it)
    auto plane_at = [&](int mm) -> double {
        const int pz = nzm - mm, from = pz * sgn > 0 ? sgn : 0;
        const double zb = (double)(pz - from) * g.t + (double)from * g.t;
        return on && fA != 0.0 ? (zb - r.sz) * duzD : 1.0e300;
    };
    int il = (int)fmin(fmax(floor((D0 + 1e-3 * g.s) * fA + (r.sz * c.ninv_t + c.nzm)), -1.0e9), 1.0e9);
    double dnext = plane_at(il + up);
    {  // (a plane within the first thousandth of the first step is met in that step)
        const double Dprev = plane_at(il + up - sgn);
        const bool back = on && fA != 0.0 && Dprev > D0;
        il -= back ? sgn : 0;
        dnext = back ? Dprev : dnext;
    }
    auto slice_off = [&](int i) -> int {  // cell offset of logical slice i, or out of the volume
        return on && (unsigned)(i + 1) <= (unsigned)g.Nz ? (i < 0 ? 0 : i) : (int)Acc::kOut;
    };

    for (;;) {
        int nsteps;
        int total;
#ifdef __HIP_DEVICE_COMPILE__
        {
            RunStep t;
            PieceRec p0, p1;
            bool has0, has1;
            bool ok = make_run_step<ALIGNED>(g, r, c, k + lane, t, p0, p1, has0, has1) && k + lane <= kmax;
            const unsigned long long bad = __ballot(!ok);
            nsteps = bad ? __ffsll((long long)bad) - 1 : 64;
            const bool in = lane < nsteps;
            const unsigned long long b0 = __ballot(in && has0), b1 = __ballot(in && has1);
            const unsigned long long below = (1ull << lane) - 1ull;
            const int pos = __popcll(b0 & below) + __popcll(b1 & below);
            total = __popcll(b0) + __popcll(b1);
            t.flags |= pos << RUN_SHIFT;
            lds->dk[lane] = t.dk;
            lds->dv[lane] = t.dv;
            lds->flags[lane] = t.flags;
            if (in && has0) lds->pieces[pos] = p0;
            if (in && has1) lds->pieces[pos + (has0 ? 1 : 0)] = p1;
            __builtin_amdgcn_wave_barrier();
        }
#else
        {
            nsteps = 64;
            total = 0;
            for (int l = 0; l < 64; ++l) {
                RunStep t;
                PieceRec p0, p1;
                bool has0, has1;
                const bool ok = make_run_step<ALIGNED>(g, r, c, k + l, t, p0, p1, has0, has1) && k + l <= kmax;
                if (!ok && nsteps == 64) nsteps = l;
                t.flags |= total << RUN_SHIFT;
                lds->dk[l] = t.dk;
                lds->dv[l] = t.dv;
                lds->flags[l] = t.flags;
                if (l < nsteps && has0) lds->pieces[total++] = p0;
                if (l < nsteps && has1) lds->pieces[total++] = p1;
            }
        }
#endif
        for (int kb = 0; kb < nsteps; kb += nb) {
            const int ke = kb + nb < nsteps ? kb + nb : nsteps;
#ifdef __HIP_DEVICE_COMPILE__
            const int pa = __builtin_amdgcn_readfirstlane(lds->flags[kb]) >> RUN_SHIFT;
            const int pb = ke < nsteps ? __builtin_amdgcn_readfirstlane(lds->flags[ke]) >> RUN_SHIFT : total;
#else
            const int pa = lds->flags[kb] >> RUN_SHIFT;
            const int pb = ke < nsteps ? lds->flags[ke] >> RUN_SHIFT : total;
#endif
            const bool cross = dnext < r.pha * lds->dk[ke - 1];
            const int zo = slice_off(il), zn = slice_off(il + sgn);
            // Crossing lanes: the step and the piece that hold the plane.  The piece is left out of the list's sums, pieces
            // from gap_end on go to the next slice, and the two parts beside the plane are gathered for themselves.
            int first_new = INT_MAX, gap_end = INT_MAX;
            bool special = false, tie = false;
            typename Acc::Q v1, v2;  // the parts
            int c1 = (int)Acc::kOut, c2 = c1;
            float l1 = 0.0f, l2 = 0.0f;
            if (any_lane(cross)) {
                int kc = (int)((dnext - D0) * g.inv_s);
                kc = kc < kb ? kb : (kc >= ke ? ke - 1 : kc);
                if (cross) {
                    const RunStep t{lds->dk[kc], lds->dv[kc], lds->flags[kc]};
                    const double Db0 = kc > 0 ? r.pha * lds->dk[kc - 1] : D0;
                    const double Dk = r.pha * t.dk, Dv = r.pha * t.dv;
                    const bool splitv = (t.flags & STEP_SPLITV) != 0;
                    tie = splitv && fabs(Dk - dnext) == fabs(Dk - Dv);
                    const bool z0 = !splitv || dnext < Dv;  // the plane lies in the first piece
                    const double a = z0 ? Db0 : Dv, b = z0 && splitv ? Dv : Dk;
                    const bool listed = (t.flags & (z0 ? STEP_OK0 : STEP_OK1)) != 0;
                    first_new = (t.flags >> RUN_SHIFT) + (!z0 && (t.flags & STEP_OK0) ? 1 : 0);
                    const bool zero = il + up == nzm;  // the z = 0 plane splits nothing: whole, by the midpoint
                    special = !zero && ((t.flags & RUN_SPECIAL) || tie);
                    const double at = zero ? ((a + b) * 0.5 < dnext ? b : a) : dnext;
                    gap_end = first_new + (listed ? 1 : 0);
                    if (listed && !special) {  // (a part of no length is not charged: its voxel may be infinite)
                        const int cb = lds->pieces[first_new].cb;
                        l1 = (float)(fmax(at - a, 0.0) * r.K);
                        l2 = (float)(fmax(b - at, 0.0) * r.K);
                        c1 = l1 > 0.0f ? cb + zo : (int)Acc::kOut;
                        c2 = l2 > 0.0f ? cb + zn : (int)Acc::kOut;
                    }
                }
                // The parts' gathers go out before the block's and are added after it (kEarly): waiting for them here, or after
                // the main loop, costs the wave a memory latency each per block (320x320x77 at 0.977 mm / 120 angles over
                // two channels 2.02 ms against 1.86; 458x458x21 at 0.598 mm / 120 angles over u16 maps 624 against
                // 590 us).  Records for which that takes registers from the gathers themselves are gathered after it
                // (u16 maps on the plane grid: 1.40 against 1.42 ms); the order of the sums is the same.
                if (any_lane(special)) {
                    // the parts from their own midpoints, off the list; with equal crossing distances the whole chord
                    // once, in place of both pieces
                    const RunStep t{lds->dk[kc], lds->dv[kc], lds->flags[kc]};
                    const bool splitv = (t.flags & STEP_SPLITV) != 0;
                    const bool z0 = !splitv || dnext < r.pha * t.dv;
                    const double uz = r.pha * dnext + r.su, uv = t.dv + r.su;
                    const double uk = plane_u(r, k + kc, g.s), ub0 = plane_u(r, k + kc - 1, g.s);
                    const Seg s1 = make_seg<false, false>(g, r, c, tie || z0 ? ub0 : uv, tie ? uk : uz, on && special, 0, false);
                    const Seg s2 = make_seg<false, false>(g, r, c, uz, z0 && splitv ? uv : uk, on && special && !tie, 0, false);
                    if (special) {
                        c1 = s1.ok ? s1.cell : (int)Acc::kOut;
                        l1 = s1.ok ? (float)s1.rr : 0.0f;
                        c2 = s2.ok ? s2.cell : (int)Acc::kOut;
                        l2 = s2.ok ? (float)s2.rr : 0.0f;
                        if (tie) {  // both pieces are left out
                            first_new = t.flags >> RUN_SHIFT;
                            gap_end = first_new + (t.flags & STEP_OK0 ? 1 : 0) + (t.flags & STEP_OK1 ? 1 : 0);
                        }
                    }
                }
                if (kEarly) {
                    acc.load(c1, v1);
                    acc.load(c2, v2);
                }
            }
            run_gaps(acc, lds->pieces, pa, pb, first_new, gap_end, zo, zn, r.K, 0);
            if (any_lane(cross)) {
                if (!kEarly) {
                    acc.load(c1, v1);
                    acc.load(c2, v2);
                }
                acc.add(v1, l1);
                acc.add(v2, l2);
                if (cross) {
                    il += sgn;
                    dnext = plane_at(il + up);
                }
            }
        }
        if (nsteps < 64) break;
        D0 = r.pha * lds->dk[63];
#ifdef __HIP_DEVICE_COMPILE__
        __builtin_amdgcn_wave_barrier();  // all reads of this table before the next fill
#endif
        k += 64;
    }
}

// The run walk in the step walk's order of additions, for sums that must come out bit for bit as the step walk's
// (traverse_table, aligned plane grids): the loss forms of the coefficient kernels, whose FP64 losses would otherwise move
// by ~1e-6 where a fit holds constant maps (FP32 sums of equal terms round one way).  The log projection takes walk_runs,
// so a loss formed from it differs from the fused one by that much.  A piece's length is rounded as (float)(|b - a| K) per
// ray; a split step adds its second piece before its first where the step walk's pipelined gather does
// (Acc::kSecondFirst); a crossing lane's first part is charged in its place and the second held and handed over where the
// step walk hands it over (before the step in which a lane that holds a piece crosses again).  Steps at the circle's
// boundary, and the rare ones with equal crossing distances, run as the step walk runs them.
// Ten vector instructions per piece and channel pair.
template <class Acc>
__host__ __device__ __forceinline__ void walk_runs_ordered(const ProjGeom& g, const RayCtx& r_in, bool active,
                                                           int kmin, int kmax, int nb, Acc& acc, OrderedLds* lds) {
#pragma clang fp contract(fast)
#ifdef __HIP_DEVICE_COMPILE__
    RayCtx r = r_in;
    r.ui = first_lane(r_in.ui);
    r.uf = first_lane(r_in.uf);
    r.vi = first_lane(r_in.vi);
    r.vf = first_lane(r_in.vf);
    r.uin = first_lane(r_in.uin);
    r.pha = first_lane(r_in.pha);
    r.dirv = first_lane(r_in.dirv);
    const int lane = threadIdx.x & 63;
    HeldPiece* hp = &lds->table.held[lane];
#else
    const RayCtx& r = r_in;
    HeldPiece* hp = &lds->table.held[0];
#endif
    const double lim_u = g.lim_u;
    const bool on = active && r.hit;
    const ChargeC c = charge_consts(g, r);
    LaneZ lz;
    lz.zA = 0.5 * r.dz * c.ninv_t;
    lz.zB = r.sz * c.ninv_t + c.nzm;
    lz.K = r.K;
    const double u0 = r.uin;
    const double v0 = (u0 - r.su) * r.dv + r.sv;
    if (!(u0 <= lim_u && u0 >= -lim_u && v0 <= lim_u && v0 >= -lim_u)) return;
    auto charge = [&](const Seg& sg) {
        typename Acc::Q q;
        acc.load(sg.ok ? sg.cell : (int)Acc::kOut, q);
        acc.add(q, sg.ok ? (float)sg.rr : 0.0f);
    };
    int k = kmin;
    double b0;  // the previous plane, relative to the source
    if (k <= 1) {
        charge(make_seg<false, false>(g, r, c, r.ui, u0, on, 0, false));
        k = 1;
        b0 = u0 - r.su;
    } else {
        b0 = plane_u(r, k - 1, g.s) - r.su;
    }
    const double dt = r.dirz * g.t, inv_t = g.inv_t;
    const double fA = r.pha * r.dz * c.ninv_t;
    const double duzD = r.pha * r.duz;
    const int up = fA > 0.0 ? 1 : 0, sgn = fA > 0.0 ? 1 : -1;
    const int nzm = (int)c.nzm;
    auto plane_at = [&](int mm) -> double {  // as in walk_runs
        const int pz = nzm - mm, from = pz * sgn > 0 ? sgn : 0;
        const double zb = (double)(pz - from) * g.t + (double)from * g.t;
        return on && fA != 0.0 ? (zb - r.sz) * duzD : 1.0e300;
    };
    const double D0 = b0 * r.pha;
    int il = (int)fmin(fmax(floor((D0 + 1e-3 * g.s) * fA + (r.sz * c.ninv_t + c.nzm)), -1.0e9), 1.0e9);
    double dnext = plane_at(il + up);
    {
        const double Dprev = plane_at(il + up - sgn);
        const bool back = on && fA != 0.0 && Dprev > D0;
        il -= back ? sgn : 0;
        dnext = back ? Dprev : dnext;
    }
    auto slice_off = [&](int i) -> int {
        return on && (unsigned)(i + 1) <= (unsigned)g.Nz ? (i < 0 ? 0 : i) : (int)Acc::kOut;
    };
    StepRec* tab = lds->table.steps;
    bool held = false;
    auto flush = [&]() {
        const HeldPiece q = *hp;
        const bool qon = held && (q.flags & STEP_OK0) && ((q.flags & STEP_CIRC) == 0 || in_circle(r, c, q.a, q.b));
        charge(make_piece(g, r, c, lz, q.a, q.b, q.cb, qon));
        held = false;
    };

    for (;;) {
        int nsteps, total;
        unsigned long long circ;  // the steps at the circle's boundary
#ifdef __HIP_DEVICE_COMPILE__
        {
            StepRec t;
            const bool ok = make_step(g, r, c, k + lane, t) && k + lane <= kmax;
            const unsigned long long bad = __ballot(!ok);
            nsteps = bad ? __ffsll((long long)bad) - 1 : 64;
            const bool in = lane < nsteps && !(t.flags & (STEP_SKIP | STEP_CIRC));
            const bool has0 = in && (t.flags & STEP_OK0), has1 = in && (t.flags & STEP_OK1);
            circ = __ballot(lane < nsteps && (t.flags & STEP_CIRC) && !(t.flags & STEP_SKIP));
            const unsigned long long m0 = __ballot(has0), m1 = __ballot(has1);
            const unsigned long long below = (1ull << lane) - 1ull;
            const int pos = __popcll(m0 & below) + __popcll(m1 & below);
            total = __popcll(m0) + __popcll(m1);
            const double db = plane_u(r, k + lane - 1, g.s) - r.su;  // the plane before the step
            t.flags |= pos << RUN_SHIFT;
            tab[lane] = t;
            if (has1) lds->pieces[pos + (!Acc::kSecondFirst && has0 ? 1 : 0)] = OrderedPiece{fabs(t.dk - t.dv), t.cb1, 0};
            if (has0) lds->pieces[pos + (Acc::kSecondFirst && has1 ? 1 : 0)] = OrderedPiece{fabs(t.dv - db), t.cb0, 0};
            __builtin_amdgcn_wave_barrier();
        }
#else
        {
            nsteps = 64;
            total = 0;
            circ = 0;
            double db = b0;
            for (int l = 0; l < 64; ++l) {
                StepRec t;
                const bool ok = make_step(g, r, c, k + l, t) && k + l <= kmax;
                if (!ok && nsteps == 64) nsteps = l;
                const bool in = l < nsteps && !(t.flags & (STEP_SKIP | STEP_CIRC));
                if (l < nsteps && (t.flags & STEP_CIRC) && !(t.flags & STEP_SKIP)) circ |= 1ull << l;
                t.flags |= total << RUN_SHIFT;
                tab[l] = t;
                for (int q = 0; q < 2; ++q) {
                    const bool second = (q == 0) == Acc::kSecondFirst;
                    if (in && (t.flags & (second ? STEP_OK1 : STEP_OK0)))
                        lds->pieces[total++] = second ? OrderedPiece{fabs(t.dk - t.dv), t.cb1, 0}
                                                      : OrderedPiece{fabs(t.dv - db), t.cb0, 0};
                }
                db = t.dk;
            }
        }
#endif
        const double Dc = r.pha * b0;  // the plane before the chunk's first step
        for (int i = 0; i < nsteps;) {
            bool slow = (circ >> i) & 1ull;
            if (!slow) {
                int ie = i + nb < nsteps ? i + nb : nsteps;
                const unsigned long long cm = circ >> i;
#ifdef __HIP_DEVICE_COMPILE__
                if (cm) ie = min(ie, i + __ffsll((long long)cm) - 1);
#else
                if (cm) ie = std::min(ie, i + __builtin_ctzll(cm));
#endif
                // the lane's crossing in the block: its step and piece
                bool cross = dnext < r.pha * tab[ie - 1].dk;
                int kc = INT_MAX, px = INT_MAX, first_new = INT_MAX;
                float lo = 0.0f;
                bool hold = false, event = false, tie = false;
                HeldPiece hnew{0.0, 0.0, 0, 0};
                if (any_lane(cross)) {
                    if (cross) {
                        kc = (int)((dnext - Dc) * g.inv_s);
                        kc = kc < i ? i : (kc >= ie ? ie - 1 : kc);
                        const StepRec t = tab[kc];
                        const double db = kc > 0 ? tab[kc - 1].dk : b0;
                        const double dzc = r.pha * dnext;
                        const bool splitv = (t.flags & STEP_SPLITV) != 0;
                        const double chz = fabs(t.dk - dzc), chv = fabs(t.dk - t.dv);
                        const bool zero = il + up == nzm;  // the z = 0 plane splits nothing
                        const bool skip = (t.flags & STEP_SKIP) != 0;
                        event = !zero && !skip;
                        tie = event && splitv && chz != 0.0 && chz == chv;
                        const bool z0 = !splitv || chz > chv;
                        const bool has0 = !skip && (t.flags & STEP_OK0), has1 = !skip && (t.flags & STEP_OK1);
                        const int base = t.flags >> RUN_SHIFT;
                        const int i1 = base + (!Acc::kSecondFirst && has0 ? 1 : 0);
                        const int i0 = base + (Acc::kSecondFirst && has1 ? 1 : 0);
                        const double a = z0 ? db : t.dv, b = z0 ? t.dv : t.dk;  // (dv = dk without a split)
                        const bool mold = zero ? r.pha * ((a + b) * 0.5) < dnext : true;
                        // the part of the piece that stays in the old slice
                        const float part = (float)((zero ? (mold ? fabs(b - a) : 0.0) : fabs(dzc - a)) * lz.K);
                        if (z0) {  // the first piece up to the plane, the second beyond it
                            first_new = base;
                            if (has0 && mold) px = i0, lo = part;
                        } else {  // the first piece before the plane, the second up to it
                            first_new = i0 + (has0 ? 1 : 0);
                            if (has1 && mold) px = i1, lo = part;
                            if (Acc::kSecondFirst && !mold) {
                                first_new = base;
                                if (has0) px = i0, lo = (float)(fabs(t.dv - db) * lz.K);
                            }
                        }
                        hold = on && event && chz != 0.0 && !tie;
                        hnew = HeldPiece{dzc, b, z0 ? t.cb0 : t.cb1, (z0 ? has0 : has1) ? (int)STEP_OK0 : 0};
                    }
                    // (lanes with equal crossing distances: the block ends before their step, which runs as a step)
                    if (any_lane(tie)) {
                        const int cut = lanes_min(tie ? kc : INT_MAX);
                        slow = cut == i;
                        ie = cut;
                        if (kc >= ie) {
                            cross = hold = event = false;
                            px = first_new = INT_MAX;
                        }
                    }
                }
                if (!slow) {
                    const int zo = slice_off(il), zn = slice_off(il + sgn);
#ifdef __HIP_DEVICE_COMPILE__
                    int pa = __builtin_amdgcn_readfirstlane(tab[i].flags) >> RUN_SHIFT;
                    const int pb = ie < nsteps ? __builtin_amdgcn_readfirstlane(tab[ie].flags) >> RUN_SHIFT : total;
#else
                    int pa = tab[i].flags >> RUN_SHIFT;
                    const int pb = ie < nsteps ? tab[ie].flags >> RUN_SHIFT : total;
#endif
                    // A lane that holds a piece and crosses again: all held pieces, those of the block's earlier
                    // crossings among them, are handed over before that step.  (Once in a block at most: after it no
                    // lane that holds a piece crosses again in the block.)
                    if (any_lane(event && held)) {
                        const int kf = lanes_min(event && held ? kc : INT_MAX);
#ifdef __HIP_DEVICE_COMPILE__
                        const int pf = __builtin_amdgcn_readfirstlane(tab[kf].flags) >> RUN_SHIFT;
#else
                        const int pf = tab[kf].flags >> RUN_SHIFT;
#endif
                        acc.run_ordered(lds->pieces, pa, pf, px, first_new, lo, zo, zn, lz.K);
                        if (hold && kc < kf) {
                            *hp = hnew;
                            held = true;
                            hold = false;
                        }
                        flush();
                        pa = pf;
                    }
                    acc.run_ordered(lds->pieces, pa, pb, px, first_new, lo, zo, zn, lz.K);
                    if (hold) {
                        *hp = hnew;
                        held = true;
                    }
                    if (cross) {
                        il += sgn;
                        dnext = plane_at(il + up);
                    }
                    b0 = tab[ie - 1].dk;
                    i = ie;
                    continue;
                }
            }
            // one step as traverse_table runs it
            {
                const StepRec t = tab[i];
                const double dk = t.dk, dv = t.dv;
                const int flags = t.flags;
                const double zk = dk * r.dz + r.sz;
                const int zma = (int)(zk * inv_t);
                const bool hz = zma != (int)((b0 * r.dz + r.sz) * inv_t);
                if (any_lane(hz && held)) flush();
                const double zb = (zma * g.t) - ((zk < 0 && r.dirz < 0) || (zk > 0 && r.dirz > 0) ? 0.0 : dt);
                const double dzc = hz ? (zb - r.sz) * r.duz : dk;
                const bool splitv = (flags & STEP_SPLITV) != 0;
                const double chz = fabs(dk - dzc), chv = fabs(dk - dv);
                const bool splitz = hz && chz != 0.0;
                const bool tie = splitv && splitz && chz == chv;
                const bool z0 = splitz && !tie && (!splitv || chz > chv);
                const bool z1 = splitz && !tie && !z0;
                if (on && (z0 || z1)) {
                    *hp = HeldPiece{dzc, z0 ? dv : dk, z0 ? t.cb0 : t.cb1,
                                    z0 ? (flags & (STEP_OK0 | STEP_CIRC))
                                       : ((flags & STEP_OK1) ? STEP_OK0 : 0) | (flags & STEP_CIRC)};
                    held = true;
                }
                double e0 = z0 ? dzc : dv;
                const double e1 = z1 ? dzc : dk;
                int cb0 = t.cb0;
                bool on0 = on && (flags & STEP_OK0);
                bool on1 = on && !tie && (flags & STEP_OK1);
                if (tie) {
                    cb0 = span_base(g, r, c, b0, dk, t.majterm);
                    e0 = dk;
                    on0 = on && cb0 >= 0;
                }
                if ((flags & STEP_CIRC) || tie) on0 = on0 && in_circle(r, c, b0, e0);
                if (flags & STEP_CIRC) on1 = on1 && splitv && in_circle(r, c, dv, e1);
                if (splitv && Acc::kSecondFirst) charge(make_piece(g, r, c, lz, dv, e1, t.cb1, on1));
                charge(make_piece(g, r, c, lz, b0, e0, cb0, on0));
                if (splitv && !Acc::kSecondFirst) charge(make_piece(g, r, c, lz, dv, e1, t.cb1, on1));
                if (dnext < r.pha * dk) {
                    il += sgn;
                    dnext = plane_at(il + up);
                }
                b0 = dk;
                ++i;
            }
        }
        if (nsteps < 64) break;
#ifdef __HIP_DEVICE_COMPILE__
        __builtin_amdgcn_wave_barrier();  // all reads of this table before the next fill
#endif
        k += 64;
    }
    if (any_lane(held)) flush();
}

}  // namespace vcbct
