// CPU build of the slice-run walk (virtualcbct_amd/csrc/runs.h) for tests: each 64-row wave is emulated on the
// host (the wave-wide step range, slope and box entry are taken over its lanes, as the kernels do), its lanes
// walked one at a time.  Test infrastructure only.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdint>
#include <vector>

#include "runs.h"

namespace {
struct HostRunAcc {
    const uint16_t* vol;  // reference layout [z][mat][y][x]
    int N, Nz, nmat;
    double L[VCBCT_MAX_MAT];
    struct Q {
        int cell;
    };
    static constexpr int kOut = 1 << 27;
    void load(int cell, Q& q) const { q.cell = cell; }
    void add(const Q& q, float len) {
        if ((unsigned)q.cell >= (unsigned)(N * N) * (unsigned)Nz) return;
        const size_t n2 = (size_t)N * N, xy = q.cell / Nz, z = q.cell % Nz;
        for (int m = 0; m < nmat; ++m) L[m] += (double)vol[(z * nmat + m) * n2 + xy] * (double)len;
    }
    void run(const vcbct::PieceRec* p, int pa, int pb, int px, int first_new, float lo, int zo, int zn, float K) {
        for (int i = pa; i < pb; ++i) {
            Q q;
            load(p[i].cb + (i < first_new ? zo : zn), q);
            add(q, i == px ? lo : p[i].len * K);
        }
    }
    static constexpr bool kSecondFirst = true;
    void run_ordered(const vcbct::OrderedPiece* p, int pa, int pb, int px, int first_new, float lo, int zo, int zn,
                     double K) {
        for (int i = pa; i < pb; ++i) {
            Q q;
            load(p[i].cb + (i < first_new || i == px ? zo : zn), q);
            add(q, i == px ? lo : (float)(p[i].len * K));
        }
    }
};
struct FirstFirstAcc : HostRunAcc {
    static constexpr bool kSecondFirst = false;
};
struct StepAcc {
    HostRunAcc* a;
    void step(const vcbct::Seg& s0, const vcbct::Seg& s1, const vcbct::Seg& s2) {
        for (const vcbct::Seg* s : {&s0, &s1, &s2})
            if (s->ok) a->add(HostRunAcc::Q{s->cell}, (float)s->rr);
    }
};
}  // namespace

// Line integrals [angle][row][col][mat]; `runs` 0: the per-lane step walk for every wave, 1: the run walk, 2 / 3: the
// ordered run walk (a split step's second piece first / last) where the plane grid is aligned.  Returns the number of
// waves that took the run walk.
extern "C" long hr_line_integrals(int N, double s, int Nz, double t, int H, int W, int nAng, double x_reg,
                                  double y_reg, double z_reg, double pitch, double pitch_iso, double sad,
                                  double pixnum, int nmat, const double* tab, const uint16_t* vol, double* L,
                                  int runs) {
    vcbct::ProjGeom g;
    g.N = N; g.Nz = Nz; g.H = H; g.W = W; g.nAng = nAng; g.nmat = nmat;
    g.s = s; g.t = t; g.x_reg = x_reg; g.y_reg = y_reg; g.z_reg = z_reg;
    g.pitch = pitch; g.pitch_iso = pitch_iso; g.sad = sad; g.pixnum = pixnum;
    vcbct::derive_geom(g);
    long taken = 0;
#pragma omp parallel for collapse(2) schedule(dynamic) reduction(+ : taken)
    for (int a = 0; a < nAng; ++a)
        for (int jj = 0; jj < W; ++jj)
            for (int rg = 0; rg < (H + 63) / 64; ++rg) {
                vcbct::RayCtx r[64];
                bool act[64];
                int kmin = INT_MAX, kmax = INT_MIN;
                float slope = 0.0f;
                for (int l = 0; l < 64; ++l) {
                    const int j = rg * 64 + l;
                    act[l] = j < H;
                    vcbct::ray_setup(g, tab[a], tab[nAng + a], tab[2 * nAng + a], tab[3 * nAng + a], act[l] ? j : 0, jj,
                                     r[l]);
                    int lo, hi;
                    vcbct::z_step_range(g, r[l], act[l], lo, hi);
                    kmin = std::min(kmin, lo);
                    kmax = std::max(kmax, hi);
                    if (lo <= hi) slope = std::max(slope, vcbct::run_slope(r[l]));
                }
                bool same = true;
                for (int l = 1; l < 64; ++l) same = same && r[l].swap == r[0].swap;
                if (kmin > kmax) continue;
                const int nb = same && runs && (runs == 1 || g.aligned) ? vcbct::run_block_steps(g, slope) : 0;
                taken += nb > 0;
                vcbct::WalkLds lds;
                for (int l = 0; l < 64; ++l) {
                    if (!act[l]) continue;
                    FirstFirstAcc acc{vol, N, Nz, nmat, {0, 0, 0, 0, 0, 0}};
                    if (nb > 0 && runs == 2)
                        vcbct::walk_runs_ordered(g, r[l], true, kmin, kmax, nb, (HostRunAcc&)acc, &lds.ordered);
                    else if (nb > 0 && runs == 3)
                        vcbct::walk_runs_ordered(g, r[l], true, kmin, kmax, nb, acc, &lds.ordered);
                    else if (nb > 0 && g.aligned)
                        vcbct::walk_runs<true>(g, r[l], true, kmin, kmax, nb, acc, &lds.runs);
                    else if (nb > 0)
                        vcbct::walk_runs<false>(g, r[l], true, kmin, kmax, nb, acc, &lds.runs);
                    else {
                        StepAcc st{&acc};
                        vcbct::traverse_lane(g, r[l], true, kmin, kmax, st);
                    }
                    const size_t o = (size_t)a * H * W + (size_t)(H - 1 - (rg * 64 + l)) * W + jj;
                    for (int m = 0; m < nmat; ++m) L[o * nmat + m] = acc.L[m];
                }
            }
    return taken;
}
