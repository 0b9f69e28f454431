// The adjoint's scatter by voxel tiles: grad += c_ray * length over all charged segments, summed in LDS.
//
// The transposed traversal of reprojectionKernel (P/reprojectionOnGPU.cu:56-690); the reference has no adjoint.
// The ray-ordered scatter (k_adjoint_scatter) issues one global FP32 atomic per charged voxel and channel, and
// they execute beyond the XCDs' L2s at ~2.6e11 a second whatever the kernel does: 38.8 of the 54.7 ms of the
// dual-energy gradient of a 512x512x64 / 360-angle problem.  Here a block owns a tile of ST x ST voxel columns by SZ
// slices in LDS, visits every ray that crosses the tile at the angles of its group, and adds the tile to the gradient
// once at the end, so that a voxel costs one global atomic per angle group instead of one per ray.
// Measured: that scatter 38.8 -> 13.15 ms, 256x256x64 / 360 angles / one channel 11.4 -> 6.1 ms, 256x256x64 / 90 angles of
// 256x256 / two channels 2.87 -> 1.2 ms.  What bounds it now is vector issue (5.0e9 wave-instructions, 61 % of the
// cycles; a fifth of them the steps of the columns, formed anew for every tile) beside the LDS atomics (51 %).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>

#include "runs.h"
#include "vcbct_internal.h"

namespace vcbct {

constexpr int ST = kScatterSide, SZ = kScatterSlices;  // 64 KB of FP64 sums a channel; a CU's 160 KB hold two, and 16 waves' lists
constexpr int SK = 20;  // steps of a ray in a tile: at most ST + 1 voxels along the major axis, and one each side

// The xy path of the rays of one detector column at one angle (the same for all its rows), made by k_scatter_rays.
// iM = 1 / (pu - su), q1 = 1 + dv^2, M = |pu - su|; entry: the voxel column (y << 16 | x) of the lumped entry segment, or -1.
struct alignas(16) ScatterRay {
    double su, sv, dv, duv, ui, uin, iM, q1;
    int flags, nb, entry;
    float M;
};
enum { SR_LIVE = 1, SR_XMAJ = 2, SR_VMOVE = 4, SR_PHA = 8, SR_DIRV = 16 };

// Workspace: the rays' paths, then the number and the list of the columns left to the ray-ordered scatter.
static size_t scatter_ray_bytes(const ProjGeom& g) { return (size_t)g.nAng * g.W * sizeof(ScatterRay); }
size_t scatter_work_bytes(const ProjGeom& g) {
    return scatter_ray_bytes(g) + 16 + (size_t)g.nAng * g.W * sizeof(int);
}

// One thread per (angle, column).
__global__ __launch_bounds__(256) void k_scatter_rays(ProjGeom g, const double* __restrict__ tab,
                                                      ScatterRay* __restrict__ rays, int* __restrict__ listed) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= g.nAng * g.W) return;
    const int a = e / g.W, jj = e - a * g.W;
    RayCtx r;
    ray_setup(g, tab[a], tab[g.nAng + a], tab[2 * g.nAng + a], tab[3 * g.nAng + a], 0, jj, r);
    ScatterRay o;
    o.su = r.su;
    o.sv = r.sv;
    o.dv = r.dv;
    o.duv = r.duv;
    o.ui = r.ui;
    o.uin = r.uin;
    o.iM = 1.0 / (r.pu - r.su);
    o.q1 = 1.0 + r.dv * r.dv;
    o.M = (float)fabs(r.pu - r.su);
    o.entry = -1;
    o.flags = 0;
    o.nb = 0;
    // plane 0 in the box, as the walks test it
    const double u0 = r.uin, v0 = (u0 - r.su) * r.dv + r.sv;
    if (r.hit && u0 <= g.lim_u && u0 >= -g.lim_u && v0 <= g.lim_u && v0 >= -g.lim_u) {
        // Rows may differ in which box hit is the entry only where the two are equally far (a ray through a box
        // corner); two slice planes in one step need t < slope s, slope <= the volume's reach in z over the source's
        // distance.  Both are left to the ray-ordered scatter, which decides them per lane.
        const double di = (r.ui - r.su) * (r.ui - r.su) + (r.vi - r.sv) * (r.vi - r.sv);
        const double df = (r.uf - r.su) * (r.uf - r.su) + (r.vf - r.sv) * (r.vf - r.sv);
        const double near_d = fmin(fabs(r.ui - r.su), fabs(u0 - r.su));
        const int nzm = (int)g.nzm;
        const double zr = fmax((double)(nzm + 1), (double)(g.Nz - nzm)) * g.t + fabs(r.sz);
        o.nb = run_block_steps(g, (float)(zr / near_d) * 1.00001f);
        if (fabs(di - df) <= 1e-6 * (di + df) || o.nb < 1) {
            listed[4 + atomicAdd(listed, 1)] = e;
        } else {
            o.flags = SR_LIVE | (r.xmaj ? SR_XMAJ : 0) | (r.vmove ? SR_VMOVE : 0) | (r.pha > 0 ? SR_PHA : 0) |
                      (r.dirv > 0 ? SR_DIRV : 0);
            const ChargeC c = charge_consts(g, r);
            const double um = (r.ui + u0) * 0.5;
            const double vm = (um - r.su) * r.dv + r.sv;
            const int imin = (int)(vm * c.smin + c.nmaj);
            const int imaj = major_index(g, r, c, r.ui, u0);
            if ((unsigned)imaj < (unsigned)g.N && (unsigned)imin < (unsigned)g.N && um * um + vm * vm < c.rmax2)
                o.entry = r.xmaj ? imin << 16 | imaj : imaj << 16 | imin;
        }
    }
    rays[e] = o;
}

// The steps of one column in the tile (as runs.h's RunStep and piece list; pieces outside the tile left out, a piece's
// column as its index in the tile).
struct ScatterSub {
    double dv[SK], len[2 * SK];
    short at[2 * SK], flags[SK];
};

// A wave forms the steps of three neighbouring detector columns at a time, a step per lane, and then walks each column's
// rays, 64 rows at a time: a lane is one ray, walked by runs (runs.h: the lane's slice and next plane carried through
// blocks of steps that hold at most one of its plane crossings).  The column's pieces sit in the lanes of two
// registers and are broadcast from there (readlane), so that a piece is one atomic per channel and no other LDS access:
// list reads would wait for the atomics before them.
// The sums are FP64: the LDS unit takes an FP32 atomic add lane by lane (193 cycles a wave), an FP64 one 16 lanes at a
// time (8.6 cycles).  A sixteen's lanes of one address repeat its pass (two rows to a slice: 20 cycles in row order), so
// neighbouring rows, which share a slice where the rows are denser than the slices, go to different sixteens (10.5;
// `spread`: log2 of the row distance within a sixteen).
// Block (tile, slice chunk, angle group); its waves take the group's angles, or every nsplit-th three columns of one,
// from a counter.
template <int NCH, bool ALIGNED>
__global__ __launch_bounds__(512 * NCH) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_scatter_tiles(
    ProjGeom g, const double* __restrict__ tab, const ScatterRay* __restrict__ rays, const float* __restrict__ coef,
    float* __restrict__ gvox, int ntx, int nang, int nsplit, int spread) {
#pragma clang fp contract(fast)
    constexpr int PLANE = ST * ST * SZ, SW = 8 * NCH;  // waves per block
    __shared__ double acc[NCH * PLANE];
    __shared__ ScatterSub subs[SW][3];
    __shared__ int next;
    const int x0 = (int)(blockIdx.x % ntx) * ST, y0 = (int)(blockIdx.x / ntx) * ST;
    const int zc = blockIdx.y * SZ, nz = min(SZ, g.Nz - zc);
    const int nxm = (int)g.nmaj, nzm = (int)g.nzm;
    // the tile's extent [cm]; the truncated index range (-1, 0) belongs to index 0
    const double xa = ((x0 ? x0 : -1) - nxm) * g.s, xb = (x0 + ST - nxm) * g.s;
    const double ya = -((y0 + ST) - nxm) * g.s, yb = -((y0 ? y0 : -1) - nxm) * g.s;
    {
        const double nx = xa > 0 ? xa : xb < 0 ? xb : 0.0, ny = ya > 0 ? ya : yb < 0 ? yb : 0.0;
        if (nx * nx + ny * ny > g.rmax2 * 1.0001) return;  // wholly outside the circle (uniform over the block)
    }
    const int a0 = blockIdx.z * nang, a1 = min(a0 + nang, g.nAng);
    if (threadIdx.x == 0) next = 0;
    for (int i = threadIdx.x; i < NCH * PLANE; i += 64 * SW) acc[i] = 0.0;
    __syncthreads();

    const int lane = threadIdx.x & 63;
    const int sub = lane / SK, l = lane - sub * SK;  // (lanes 60 to 63: none)
    const int lrow = (lane & (63 >> spread)) << spread | lane >> (6 - spread);
    ScatterSub* SS = subs[threadIdx.x >> 6];
    const size_t nrays = (size_t)g.nAng * g.H * g.W;
    const double pixh = g.pitch_iso * (g.pixnum / g.H), ipixh = 1.0 / pixh;
    const double zreg = g.z_reg * g.pitch_iso / g.pitch;
    // the chunk's z range relative to the source's (slice 0 also takes the truncated range above it)
    const float zlf = (float)((double)(nzm - zc - nz) * g.t - g.z_reg);
    const float zhf = (float)((double)(nzm - zc + (zc == 0 ? 1 : 0)) * g.t - g.z_reg);

    for (;;) {
        int task = 0;
        if (lane == 0) task = atomicAdd(&next, 1);
        task = __builtin_amdgcn_readfirstlane(task);
        const int a = a0 + task / nsplit, part = task % nsplit;
        if (a >= a1) break;
        const double ct = ldk(tab, a), sn = ldk(tab, g.nAng + a), xc = ldk(tab, 2 * g.nAng + a),
                     yc = ldk(tab, 3 * g.nAng + a);
        int c0, c1;
        {  // the columns whose rays can cross the tile: its corners' projections, one corner per lane
            const double sx = -g.sad * sn + g.x_reg, sy = g.sad * ct + g.y_reg;
            const double ox = g.x_reg * g.pitch_iso / g.pitch, oy = g.y_reg * g.pitch_iso / g.pitch;
            const double ex = (lane & 1 ? xb : xa) - sx, ey = (lane & 2 ? yb : ya) - sy;
            const double mu = ((ox - sx) * -sn + (oy - sy) * ct) / (ex * -sn + ey * ct);
            const double q = (sx + mu * ex - ox) * ct + (sy + mu * ey - oy) * sn;
            float lo = (float)(q * ipixh - xc), hi = lo;
#pragma unroll
            for (int o = 1; o <= 2; o <<= 1) {
                lo = fminf(lo, __shfl_xor(lo, o, 64));
                hi = fmaxf(hi, __shfl_xor(hi, o, 64));
            }
            c0 = __builtin_amdgcn_readfirstlane(max((int)floorf(fmaxf(lo, -1e6f) - 0.02f), 0));
            c1 = __builtin_amdgcn_readfirstlane(min((int)ceilf(fminf(hi, 1e6f) + 0.02f), g.W - 1));
        }
        for (int cb = c0 + 3 * part; cb <= c1; cb += 3 * nsplit) {
            __builtin_amdgcn_wave_barrier();  // all reads of the last columns' steps before this fill
            // ---- the steps of three columns
            int k0, total, nsteps, ecell, j0, j1;
            bool parts;  // a step of the column has RUN_SPECIAL
            {
                const ScatterRay R = rays[(size_t)a * g.W + min(cb + sub, c1)];
                const bool live = sub < 3 && cb + sub <= c1 && (R.flags & SR_LIVE);
                RayCtx r;
                r.su = R.su;
                r.sv = R.sv;
                r.dv = R.dv;
                r.duv = R.duv;
                r.uin = R.uin;
                r.pha = R.flags & SR_PHA ? 1.0 : -1.0;
                r.dirv = R.flags & SR_DIRV ? 1.0 : -1.0;
                r.xmaj = (R.flags & SR_XMAJ) != 0;
                r.vmove = (R.flags & SR_VMOVE) != 0;
                ChargeC c = charge_consts(g, r);
                c.mstride = 1 << 16;  // pieces name their (minor, major) voxel column
                c.majmul = 1;
                // the tile's columns are minor + 16 major or the other way round
                const int m0 = r.xmaj ? y0 : x0, u0 = r.xmaj ? x0 : y0;
                auto place = [&](int cbase) -> int {
                    const int lm = (cbase >> 16) - m0, lu = (cbase & 0xffff) - u0;
                    return ((lm | lu) & ~(ST - 1)) == 0 ? (r.xmaj ? lm * ST + lu : lu * ST + lm) : -1;
                };
                const double ua = r.xmaj ? xa : ya, ub = r.xmaj ? xb : yb;
                const double t1 = (r.pha > 0 ? ua - r.uin : r.uin - ub) * g.inv_s;
                const double t2 = (r.pha > 0 ? ub - r.uin : r.uin - ua) * g.inv_s;
                k0 = max((int)floor(t1 - 1e-6) + 1, 1);
                nsteps = live ? max(min((int)ceil(t2 + 1e-6) - k0 + 1, SK), 0) : 0;
                RunStep t;
                PieceRec p0, p1;
                bool has0 = false, has1 = false;
                const bool in = make_run_step<ALIGNED>(g, r, c, k0 + l, t, p0, p1, has0, has1) && l < nsteps;
                p0.cb = place(p0.cb);
                p1.cb = place(p1.cb);
                has0 = in && has0 && p0.cb >= 0;
                has1 = in && has1 && p1.cb >= 0;
                const int sh = min(sub, 2) * SK;
                const unsigned below = (1u << l) - 1u, all = (1u << SK) - 1u;
                const unsigned h0 = (unsigned)(__ballot(has0) >> sh) & all, h1 = (unsigned)(__ballot(has1) >> sh) & all;
                nsteps = __popc((unsigned)(__ballot(in) >> sh) & all);  // (the walk ends where it leaves the box)
                parts = ((unsigned)(__ballot(in && (t.flags & RUN_SPECIAL)) >> sh) & all) != 0;
                const int pos = __popc(h0 & below) + __popc(h1 & below);
                total = __popc(h0) + __popc(h1);
                if (sub < 3) {
                    ScatterSub* S = SS + sub;
                    S->dv[l] = t.dv;
                    // (a step whose piece lies in another tile keeps its mark: parts are formed by their midpoints)
                    S->flags[l] = (short)((t.flags & (STEP_SPLITV | RUN_SPECIAL)) | (has0 ? STEP_OK0 : 0) |
                                          (has1 ? STEP_OK1 : 0) | pos << RUN_SHIFT);
                    if (has0) {
                        S->len[pos] = p0.len;
                        S->at[pos] = (short)p0.cb;
                    }
                    if (has1) {
                        S->len[pos + (has0 ? 1 : 0)] = p1.len;
                        S->at[pos + (has0 ? 1 : 0)] = (short)p1.cb;
                    }
                }
                ecell = live && R.entry >= 0
                            ? place(r.xmaj ? R.entry : (int)((unsigned)R.entry << 16 | (unsigned)R.entry >> 16))
                            : -1;
                // the rows whose rays can be in the chunk's slices within these steps
                const double D0 = (plane_u(r, k0 - 1, g.s) - r.su) * r.pha;
                // (FP32: off by less than the fiftieth of a row that is added on either side)
                const float Da = (float)(ecell >= 0 ? fmin(D0, (R.ui - r.su) * r.pha) : D0);
                const float Db = (float)(D0 + (nsteps + 1) * g.s);
                const float qa = R.M * __builtin_amdgcn_rcpf(Da), qb = R.M * __builtin_amdgcn_rcpf(Db);
                const float pl = zlf * (zlf > 0.0f ? qb : qa), ph = zhf * (zhf > 0.0f ? qa : qb);  // pz - sz
                const float row0 = (float)((zreg - g.z_reg) * ipixh - yc), ip = (float)ipixh;
                j0 = (int)fminf(fmaxf(floorf(row0 - ph * ip - 0.02f), 0.0f), (float)g.H);
                j1 = (int)fmaxf(fminf(ceilf(row0 - pl * ip + 0.02f), (float)(g.H - 1)), -1.0f);
                // (a part of a piece that the tile does not list can have its own midpoint in the tile, or in the circle)
                if (!(total > 0 || parts || ecell >= 0)) j1 = j0 - 1;
                __builtin_amdgcn_wave_barrier();
            }
            // ---- each column's rays
            const int nc = min(c1 - cb + 1, 3);
            for (int q = 0; q < nc; ++q) {
                const int cj0 = __builtin_amdgcn_readlane(j0, q * SK), cj1 = __builtin_amdgcn_readlane(j1, q * SK);
                if (cj1 < cj0) continue;
                const int ck0 = __builtin_amdgcn_readlane(k0, q * SK), ctot = __builtin_amdgcn_readlane(total, q * SK);
                const int ns = __builtin_amdgcn_readlane(nsteps, q * SK), ce = __builtin_amdgcn_readlane(ecell, q * SK);
                const int col = cb + q;
                const ScatterRay* RP = rays + ((size_t)a * g.W + col);
                const ScatterSub* S = SS + q;
                const int rf = ldk(&RP->flags, 0), nb = ldk(&RP->nb, 0);
                RayCtx r;
                r.su = ldk(&RP->su, 0);
                r.sv = ldk(&RP->sv, 0);
                r.dv = ldk(&RP->dv, 0);
                r.uin = ldk(&RP->uin, 0);
                r.pha = rf & SR_PHA ? 1.0 : -1.0;
                r.xmaj = (rf & SR_XMAJ) != 0;
                r.sz = g.z_reg;
                const double q1 = ldk(&RP->q1, 0), iM = ldk(&RP->iM, 0);
                const ChargeC c = charge_consts(g, r);
                const double D0 = (plane_u(r, ck0 - 1, g.s) - r.su) * r.pha;
                // lane p: piece p
                const double plen = lane < 2 * SK ? S->len[lane] : 0.0;
                const int pat = lane < 2 * SK ? S->at[lane] : 0;
                auto piece_len = [&](int p) -> double {
                    int2 q = __builtin_bit_cast(int2, plen);
                    q.x = __builtin_amdgcn_readlane(q.x, p);
                    q.y = __builtin_amdgcn_readlane(q.y, p);
                    return __builtin_bit_cast(double, q);
                };
                for (int jr = cj0; jr <= cj1; jr += 64) {
                    const int j = jr + lrow;
                    const bool on = j <= cj1;
                    double cm[NCH];
                    bool any = false;
#pragma unroll
                    for (int m = 0; m < NCH; ++m) {
                        cm[m] = on ? ldg(coef, (size_t)m * nrays + ((size_t)a * g.W + col) * g.H + j) : 0.0f;
                        any = any || cm[m] != 0.0;
                    }
                    if (!__any(any)) continue;
                    const double pz = -(yc + j) * g.pitch_iso * (g.pixnum / g.H) + zreg;
                    r.dz = (pz - r.sz) * iM;
                    {  // the length per unit of u: the root in FP32 and one Newton step in FP64 (to ~1e-14)
                        const double qq = q1 + r.dz * r.dz;
                        const float h = __builtin_amdgcn_rsqf((float)qq);
                        const double k = (double)((float)qq * h);
                        const double K = k + (qq - k * k) * (double)(0.5f * h);
#pragma unroll
                        for (int m = 0; m < NCH; ++m) cm[m] *= K;
                    }
                    // adds len c at byte `at` of the tile (negative: nowhere)
                    auto add = [&](int at, double len) {
                        if (at < 0) return;
                        double* p = (double*)((char*)acc + at);
#pragma unroll
                        for (int m = 0; m < NCH; ++m)
                            __hip_atomic_fetch_add(p + m * PLANE, cm[m] * len, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_WORKGROUP);
                    };
                    // takes it back (not of an infinite coefficient: the voxel keeps its infinity)
                    auto take = [&](int at, double len) {
                        if (at < 0) return;
                        double* p = (double*)((char*)acc + at);
#pragma unroll
                        for (int m = 0; m < NCH; ++m)
                            __hip_atomic_fetch_add(p + m * PLANE, fabs(cm[m]) <= 1.0e300 ? -cm[m] * len : 0.0,
                                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    };
                    // a segment [ua, ub] of tile column `at`, or of its own midpoint's, as the walks form them (make_seg)
                    auto segment = [&](double ua, double ub, int at) {
                        const double um = (ua + ub) * 0.5, d = um - r.su;
                        const double vm = d * r.dv + r.sv, zm = d * r.dz + r.sz;
                        const int zz = (int)(zm * c.ninv_t + c.nzm);
                        if (at < 0) {
                            const int imin = (int)(vm * c.smin + c.nmaj), imaj = major_index(g, r, c, ua, ub);
                            const int lx = (r.xmaj ? imaj : imin) - x0, ly = (r.xmaj ? imin : imaj) - y0;
                            at = (unsigned)imaj < (unsigned)g.N && (unsigned)imin < (unsigned)g.N &&
                                         ((lx | ly) & ~(ST - 1)) == 0 && um * um + vm * vm < c.rmax2
                                     ? ly * ST + lx
                                     : -1;
                        }
                        add(at >= 0 && (unsigned)(zz - zc) < (unsigned)nz ? at * (SZ * 8) + (zz - zc) * 8 : -1,
                            fabs(ub - ua));
                    };
                    if (ce >= 0 && on) segment(ldk(&RP->ui, 0), r.uin, ce);
                    // the lane's slice and next slice plane at the first step (as walk_runs)
                    const double fA = r.pha * r.dz * c.ninv_t;
                    // pha / dz, a rounding off at most (dz = 0: not used)
                    double duzD = __builtin_amdgcn_rcp(r.dz);
                    duzD = fma(fma(-r.dz, duzD, 1.0), duzD, duzD);
                    duzD = fma(fma(-r.dz, duzD, 1.0), duzD, duzD) * r.pha;
                    const int up = fA > 0.0 ? 1 : 0, sgn = fA > 0.0 ? 1 : -1;
                    auto plane_at = [&](int mm) -> double {
                        const int p = nzm - mm;
                        const double zb = p * sgn > 0 ? (double)(p - sgn) * g.t + (double)sgn * g.t : (double)p * g.t;
                        return on && fA != 0.0 ? (zb - r.sz) * duzD : 1.0e300;
                    };
                    const double fB = r.sz * c.ninv_t + c.nzm;
                    int il = (int)floor((D0 + 1e-3 * g.s) * fA + fB);  // (saturates far outside the volume)
                    double dnext = plane_at(il + up);
                    // (a plane within the first thousandth of the first step is met in that step)
                    if (__any(on && (int)floor(D0 * fA + fB) != il)) {
                        const double Dprev = plane_at(il + up - sgn);
                        if (on && fA != 0.0 && Dprev > D0) {
                            il -= sgn;
                            dnext = Dprev;
                        }
                    }
                    auto slice_off = [&](int i) -> int {  // the slice's offset in the chunk (bytes), or far below zero
                        const int z = (i < 0 ? 0 : i) - zc;
                        return on && i >= -1 && i < g.Nz && (unsigned)z < (unsigned)nz ? z * 8 : INT_MIN;
                    };
                    auto pos_of = [&](int k) -> double { return (plane_u(r, k, g.s) - r.su) * r.pha; };
                    for (int kb = 0; kb < ns; kb += nb) {
                        const int ke = min(kb + nb, ns);
                        const int pa = kb ? __builtin_amdgcn_readfirstlane((int)S->flags[kb]) >> RUN_SHIFT : 0;
                        const int pb = ke < ns ? __builtin_amdgcn_readfirstlane((int)S->flags[ke]) >> RUN_SHIFT : ctot;
                        const bool cross = dnext < pos_of(ck0 + ke - 1);
                        const int zo = slice_off(il), zn = slice_off(il + sgn);
                        // Crossing lanes: pieces from first_new on go to the next slice.  The piece that holds the plane is
                        // among those before, and its part beyond the plane is moved over in FP64: both slices are charged
                        // (a piece that lies in one of them goes there whole).  Where parts go by their own midpoints, the
                        // pieces [first_new, gap_end) are left out instead; done so in every block, two instructions a
                        // piece, the scatter of 256x256x64 / 360 angles takes 6.11 ms against 5.92.
                        int first_new = INT_MAX, gap_end = INT_MAX;
                        bool special = false;
                        if (cross) {
                            int kc = (int)((dnext - D0) * g.inv_s);
                            kc = kc < kb ? kb : (kc >= ke ? ke - 1 : kc);
                            const int fl = S->flags[kc];
                            const double Dk = pos_of(ck0 + kc), Dv = r.pha * S->dv[kc];
                            const bool splitv = (fl & STEP_SPLITV) != 0;
                            const bool tie = splitv && fabs(Dk - dnext) == fabs(Dk - Dv);
                            const bool z0 = !splitv || dnext < Dv;
                            const double ba = z0 ? pos_of(ck0 + kc - 1) : Dv, be = z0 && splitv ? Dv : Dk;
                            const bool listed = (fl & (z0 ? STEP_OK0 : STEP_OK1)) != 0;
                            const bool zero = il + up == nzm;  // the z = 0 plane splits nothing: whole, by the midpoint
                            special = !zero && ((fl & RUN_SPECIAL) || tie);
                            first_new = (fl >> RUN_SHIFT) + (!z0 && (fl & STEP_OK0) ? 1 : 0);
                            gap_end = first_new + (listed ? 1 : 0);
                            if (special) {
                                // the parts from their own midpoints; with equal crossing distances the whole chord once,
                                // in place of both pieces
                                const double uz = r.pha * dnext + r.su, uv = S->dv[kc] + r.su;
                                const double uk = plane_u(r, ck0 + kc, g.s), ub0 = plane_u(r, ck0 + kc - 1, g.s);
                                segment(tie || z0 ? ub0 : uv, tie ? uk : uz, -1);
                                if (!tie) segment(uz, z0 && splitv ? uv : uk, -1);
                                if (tie) {
                                    first_new = fl >> RUN_SHIFT;
                                    gap_end = first_new + (fl & STEP_OK0 ? 1 : 0) + (fl & STEP_OK1 ? 1 : 0);
                                }
                            } else if (listed) {
                                const double at = zero ? ((ba + be) * 0.5 < dnext ? be : ba) : dnext;
                                if (at > ba) {
                                    if (be > at) {
                                        const int cell = S->at[first_new] * (SZ * 8);
                                        add(cell + zn, be - at);
                                        take(cell + zo, be - at);
                                    }
                                    ++first_new;
                                }
                                gap_end = first_new;
                            }
                        }
                        if (!__any(special)) {
                            for (int p = pa; p < pb; ++p)
                                add(__builtin_amdgcn_readlane(pat, p) * (SZ * 8) + (p < first_new ? zo : zn), piece_len(p));
                        } else {
                            for (int p = pa; p < pb; ++p)
                                add(__builtin_amdgcn_readlane(pat, p) * (SZ * 8) +
                                        (p < first_new ? zo : p >= gap_end ? zn : INT_MIN),
                                    piece_len(p));
                        }
                        if (cross) {
                            il += sgn;
                            dnext = plane_at(il + up);
                        }
                    }
                }
            }
        }
    }
    __syncthreads();
    const size_t nvox = (size_t)g.N * g.N * g.Nz;
    for (int i = threadIdx.x; i < NCH * PLANE; i += 64 * SW) {
        const float v = (float)acc[i];
        const int z = i % SZ, x = x0 + i / SZ % ST, y = y0 + i / (SZ * ST) % ST, m = i / PLANE;
        if (v != 0.0f && z < nz && x < g.N && y < g.N)
            atomicAdd(gvox + m * nvox + ((size_t)y * g.N + x) * g.Nz + zc + z, v);
    }
}

int launch_scatter_rays(const ProjGeom& g, const double* tables, void* work, hipStream_t st, const int** listed) {
    int* li = (int*)((char*)work + scatter_ray_bytes(g));
    *listed = li;
    int rc = launch_zero(li, 16, st);
    if (rc) return rc;
    hipLaunchKernelGGL(k_scatter_rays, dim3((unsigned)(((size_t)g.nAng * g.W + 255) / 256)), dim3(256), 0, st, g,
                       tables, (ScatterRay*)work, li);
    VCBCT_HIP(hipGetLastError());
    return 0;
}

// Channels go two at a time (their LDS).
int launch_scatter_tiles(const ProjGeom& g, const double* tables, const void* work, const float* coef, int nch,
                         float* gvox, hipStream_t st) {
    const int nt = (g.N + ST - 1) / ST, nzc = (g.Nz + SZ - 1) / SZ;
    const int nang = scatter_angles(g), waves = nch > 1 ? 16 : 8;
    // columns are split where a block's waves would get fewer than four tasks each
    const double cols = 1.3 * ST * g.s / (g.pitch_iso * (g.pixnum / g.H)) + 2.0;  // a tile's, about
    const int nsplit = (int)std::max(1.0, std::min(std::ceil(4.0 * waves / nang), std::min(cols, 1.0e6) / 3.0));
    const double rps = g.t / (g.pitch_iso * (g.pixnum / g.H));  // rows per slice
    const int spread = rps < 1.0 ? 0 : rps < 3.0 ? 1 : 2;
    const size_t nrays = (size_t)g.nAng * g.H * g.W, nvox = (size_t)g.N * g.N * g.Nz;
    const dim3 grid((unsigned)(nt * nt), (unsigned)nzc, (unsigned)((g.nAng + nang - 1) / nang));
    const ScatterRay* rays = (const ScatterRay*)work;
    for (int m = 0; m < nch; m += 2) {
        const float* c = coef + (size_t)m * nrays;
        float* o = gvox + (size_t)m * nvox;
#define VCBCT_LAUNCH_TILES(C, A) \
    hipLaunchKernelGGL((k_scatter_tiles<C, A>), grid, dim3(512 * C), 0, st, g, tables, rays, c, o, nt, nang, nsplit, spread)
        if (nch - m >= 2) {
            if (g.aligned) VCBCT_LAUNCH_TILES(2, true);
            else VCBCT_LAUNCH_TILES(2, false);
        } else {
            if (g.aligned) VCBCT_LAUNCH_TILES(1, true);
            else VCBCT_LAUNCH_TILES(1, false);
        }
#undef VCBCT_LAUNCH_TILES
    }
    VCBCT_HIP(hipGetLastError());
    return 0;
}

}  // namespace vcbct
