// CPU build of the walks (virtualcbct_amd/csrc/traverse.h, runs.h) with the 64 lanes of a wave stepped together: each lane is
// a fibre that runs to the next wave-wide question, which is answered when all have reached it.  Line integrals are FP32
// sums as the kernels form them, so that their order shows.  Beside it, the host-side rules that choose a kernel.  Test
// infrastructure only.
#include <hip/hip_runtime.h>
#include <ucontext.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <functional>
#include <vector>

namespace {
struct Fibres {
    static constexpr int kLanes = 64;
    static constexpr size_t kStack = 256 * 1024;
    ucontext_t home, lane[kLanes];
    std::vector<char> stacks = std::vector<char>(kLanes * kStack);
    std::function<void(int)> body;
    int at = 0, waiting = 0, running = 0;
    bool any = false, any_answer = false;
    int least = INT_MAX, least_answer = INT_MAX;
    long questions = 0;
    bool done[kLanes];
    static Fibres* self;
    static void entry() {
        self->body(self->at);
        self->done[self->at] = true;
        --self->running;
        for (;;) swapcontext(&self->lane[self->at], &self->home);
    }
    void run(std::function<void(int)> f) {
        self = this;
        body = std::move(f);
        running = kLanes;
        for (int l = 0; l < kLanes; ++l) {
            done[l] = false;
            getcontext(&lane[l]);
            lane[l].uc_stack.ss_sp = &stacks[l * kStack];
            lane[l].uc_stack.ss_size = kStack;
            lane[l].uc_link = nullptr;
            makecontext(&lane[l], entry, 0);
        }
        while (running) {
            waiting = 0;
            any = false;
            least = INT_MAX;
            for (at = 0; at < kLanes; ++at)
                if (!done[at]) swapcontext(&home, &lane[at]);
            if (waiting && waiting != kLanes) abort();  // a wave-wide question that not every lane reached
            any_answer = any;
            least_answer = least;
            ++questions;
        }
    }
    void ask() {
        ++waiting;
        swapcontext(&lane[at], &home);
    }
};
Fibres* Fibres::self = nullptr;
bool host_any(bool b) {
    Fibres* f = Fibres::self;
    f->any = f->any || b;
    f->ask();
    return f->any_answer;
}
int host_min(int v) {
    Fibres* f = Fibres::self;
    f->least = std::min(f->least, v);
    f->ask();
    return f->least_answer;
}
}  // namespace
#define VCBCT_HOST_ANY_LANE host_any
#define VCBCT_HOST_LANES_MIN host_min
#include "runs.h"

namespace {
struct Sums {
    const uint16_t* vol;  // [z][mat][y][x]
    int N, Nz, nmat;
    float L[VCBCT_MAX_MAT] = {0, 0, 0, 0, 0, 0};
    void charge(int cell, float len) {
        if ((unsigned)cell >= (unsigned)(N * N) * (unsigned)Nz) return;
        const size_t n2 = (size_t)N * N, xy = cell / Nz, z = cell % Nz;
        for (int m = 0; m < nmat; ++m) L[m] = std::fma((float)vol[(z * nmat + m) * n2 + xy], len, L[m]);
    }
};
// The ordered walk's sums (forward.hip, OrderedAcc).
template <bool SF>
struct Ordered : Sums {
    struct Q {
        int cell;
    };
    static constexpr int kOut = 1 << 27;
    static constexpr bool kSecondFirst = SF;
    void load(int cell, Q& q) const { q.cell = cell; }
    void add(const Q& q, float len) { charge(q.cell, len); }
    void run_ordered(const vcbct::OrderedPiece* p, int pa, int pb, int px, int first_new, float lo, int zo, int zn,
                     double K) {
        for (int i = pa; i < pb; ++i)
            charge(p[i].cb + (i < first_new || i == px ? zo : zn), i == px ? lo : (float)(p[i].len * K));
    }
};
// The step walk's: a step's segments in their order (FP32 maps), or its first one with the next step (the others).
template <bool SF>
struct Step : Sums {
    vcbct::Seg held{0, 0.0, false};
    void one(const vcbct::Seg& s) {
        if (s.ok) charge(s.cell, (float)s.rr);
    }
    void step(const vcbct::Seg& a, const vcbct::Seg& b, const vcbct::Seg& c) {
        one(SF ? held : a);
        one(b);
        one(c);
        held = a;
    }
    void finish() {
        if (SF) one(held);
    }
};

vcbct::ProjGeom geom(int N, double s, int Nz, double t, int H, int W, int nAng, double x_reg, double y_reg, double z_reg,
                     double pitch, double pitch_iso, double sad, double pixnum, int nmat) {
    vcbct::ProjGeom g;
    g.N = N; g.Nz = Nz; g.H = H; g.W = W; g.nAng = nAng; g.nmat = nmat;
    g.s = s; g.t = t; g.x_reg = x_reg; g.y_reg = y_reg; g.z_reg = z_reg;
    g.pitch = pitch; g.pitch_iso = pitch_iso; g.sad = sad; g.pixnum = pixnum;
    vcbct::derive_geom(g);
    return g;
}

struct Wave {
    vcbct::RayCtx r[64];
    bool act[64], same = true;
    int lo[64], hi[64], kmin = INT_MAX, kmax = INT_MIN;
    float all = 0.0f;  // the steepest active lane that meets the box (the ordered walk's block length)
    Wave(const vcbct::ProjGeom& g, const double* tab, int a, int jj, int rg) {
        for (int l = 0; l < 64; ++l) {
            const int j = rg * 64 + l;
            act[l] = j < g.H;
            vcbct::ray_setup(g, tab[a], tab[g.nAng + a], tab[2 * g.nAng + a], tab[3 * g.nAng + a], act[l] ? j : 0, jj, r[l]);
            vcbct::z_step_range(g, r[l], act[l], lo[l], hi[l]);
            kmin = std::min(kmin, lo[l]);
            kmax = std::max(kmax, hi[l]);
            if (act[l] && r[l].hit) all = std::max(all, vcbct::run_slope(r[l]));
            same = same && r[l].swap == r[0].swap;
        }
    }
};

template <bool SF>
void walk_both(const vcbct::ProjGeom& g, Fibres& fib, const Wave& w, int nb, const uint16_t* vol, float* a, float* b) {
    std::vector<vcbct::WalkLds> lds(64);
    fib.run([&](int l) {
        Ordered<SF> acc;
        acc.vol = vol, acc.N = g.N, acc.Nz = g.Nz, acc.nmat = g.nmat;
        vcbct::walk_runs_ordered(g, w.r[l], w.act[l], w.kmin, w.kmax, nb, acc, &lds[l].ordered);
        std::copy(acc.L, acc.L + g.nmat, a + l * g.nmat);
    });
    fib.run([&](int l) {
        Step<SF> acc;
        acc.vol = vol, acc.N = g.N, acc.Nz = g.Nz, acc.nmat = g.nmat;
        vcbct::traverse_lane(g, w.r[l], w.act[l], w.kmin, w.kmax, acc, &lds[l].table);
        acc.finish();
        std::copy(acc.L, acc.L + g.nmat, b + l * g.nmat);
    });
}
}  // namespace

// Rays whose FP32 sums differ in any bit between the ordered run walk and the step table's, over every wave that can take
// both (second_first: the accumulators' order); counts[0] the rays compared, counts[1] the slice crossings that the waves
// asked about, as a measure of what was run.
extern "C" long hw_ordered_differences(int N, double s, int Nz, double t, int H, int W, int nAng, double x_reg,
                                       double y_reg, double z_reg, double pitch, double pitch_iso, double sad,
                                       double pixnum, int nmat, const double* tab, const uint16_t* vol,
                                       int second_first, long* counts) {
    const vcbct::ProjGeom g = geom(N, s, Nz, t, H, W, nAng, x_reg, y_reg, z_reg, pitch, pitch_iso, sad, pixnum, nmat);
    Fibres fib;
    std::vector<float> a(64 * nmat), b(64 * nmat);
    long differ = 0;
    counts[0] = counts[1] = 0;
    for (int an = 0; an < nAng; ++an)
        for (int jj = 0; jj < W; ++jj)
            for (int rg = 0; rg < (H + 63) / 64; ++rg) {
                const Wave w(g, tab, an, jj, rg);
                const int nb = vcbct::run_block_steps(g, w.all);
                if (w.kmin > w.kmax || !w.same || nb < 1 || !g.aligned) continue;
                if (second_first) walk_both<true>(g, fib, w, nb, vol, a.data(), b.data());
                else walk_both<false>(g, fib, w, nb, vol, a.data(), b.data());
                for (int l = 0; l < 64; ++l)
                    if (w.act[l]) {
                        ++counts[0];
                        differ += !std::equal(&a[l * nmat], &a[l * nmat] + nmat, &b[l * nmat]);
                    }
            }
    counts[1] = fib.questions;
    return differ;
}

// Row groups that rows_miss turns away: told in counts[0], and among them the lanes that charge a segment (returned).
extern "C" long hw_rows_miss_charged(int N, double s, int Nz, double t, int H, int W, int nAng, double x_reg, double y_reg,
                                     double z_reg, double pitch, double pitch_iso, double sad, double pixnum,
                                     const double* tab, long* counts) {
    const vcbct::ProjGeom g = geom(N, s, Nz, t, H, W, nAng, x_reg, y_reg, z_reg, pitch, pitch_iso, sad, pixnum, 1);
    struct Count {
        long n = 0;
        void step(const vcbct::Seg& a, const vcbct::Seg& b, const vcbct::Seg& c) { n += a.ok + b.ok + c.ok; }
    };
    long bad = 0;
    counts[0] = counts[1] = 0;
    for (int an = 0; an < nAng; ++an)
        for (int jj = 0; jj < W; ++jj)
            for (int j0 = 0; j0 < H; j0 += 64) {
                const int j1 = std::min(j0 + 63, H - 1);
                ++counts[1];
                if (!vcbct::rows_miss(g, tab[3 * nAng + an], j0, j1)) continue;
                ++counts[0];
                const Wave w(g, tab, an, jj, j0 / 64);
                for (int l = 0; l <= j1 - j0; ++l) {
                    Count c;
                    vcbct::traverse_lane(g, w.r[l], true, w.lo[l], w.hi[l], c);
                    bad += c.n > 0;
                }
            }
    return bad;
}

extern "C" int hw_scatter_by_tiles(int N, double s, int Nz, double t, int H, int W, int nAng, int nch) {
    return vcbct::scatter_by_tiles(geom(N, s, Nz, t, H, W, nAng, 0, 0, 0, 0.05, 0.032509752, 100.0, 800.0, 6), nch);
}
extern "C" int hw_thin(int N, double s, int Nz, double t, int H, int W) {
    return geom(N, s, Nz, t, H, W, 1, 0, 0, 0, 0.05, 0.032509752, 100.0, 800.0, 6).thin;
}
