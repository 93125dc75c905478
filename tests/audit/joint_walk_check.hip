// joint_walk_check.hip -- CPU check of the cone kernel's segment-sum walk as a wave runs it.  TEST INFRASTRUCTURE.
//
// The kernel walks both directions of a destination together, and a lane goes on with its wave after its own
// walks have ended.  On random lines (water, lung, bone, air and empty runs, TERMA with zero runs, a first sample that
// dwarfs the rest, lines of one sample) and radial tables that end inside the line or behind it, ramp_walk<true, true> with
// extra rounds after a lane's own end is compared with the walks' sums in FP64, sample by sample, over the same
// centres and with the same exits.  The tables are laid out as the kernel lays them out in LDS (U + 4 lookup
// entries, ramp_cells), each beside an unmapped page, behind it or before it in turn, so that an index out of
// its bounds ends the program.
//
// Tolerance: the walk looks F up at the FP32 rounding of a coordinate y <= c_{n-1}, so one F is off by at most
// ulp(c_{n-1}) / 2 times the TERMA step there, which is no more than the line's largest TERMA.  Summed by parts over
// the radii, those errors are weighed with the changes of the slope, 2 max(sigma) in sum for a row of either sign of
// curvature.  A direction is thus within max(sigma) max(T) ulp(c_{n-1}); twice that bounds also the FP64
// rounding.
//   joint_walk_check [lines] [seed]
// This file includes endtoend_amd/csrc/beam.hip and calls its functions on the host.  Prints one JSON line of
// counts and exits 1 on any mismatch.
#include "../../endtoend_amd/csrc/beam.hip"

#include <sys/mman.h>
#include <unistd.h>

#include <cinttypes>
#include <random>

namespace {

// n entries ending at an unmapped page (behind) or starting after one.
template <class T>
struct Fenced {
    char* base = nullptr;
    size_t bytes = 0;
    T* p = nullptr;
    Fenced(size_t n, bool behind) {
        const size_t page = (size_t)sysconf(_SC_PAGESIZE), need = (n * sizeof(T) + page - 1) / page * page;
        bytes = need + page;
        base = static_cast<char*>(mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
        if (base == MAP_FAILED || mprotect(behind ? base + need : base, page, PROT_NONE) != 0) std::abort();
        p = reinterpret_cast<T*>(behind ? base + need - n * sizeof(T) : base + page);
    }
    ~Fenced() { munmap(base, bytes); }
    Fenced(const Fenced&) = delete;
    Fenced& operator=(const Fenced&) = delete;
};

// A lane whose wave goes on for `left` rounds after its own end.
struct LateLane {
    static inline int left = 0;
    static bool any(bool x) { return x || left-- > 0; }
};

struct Table {
    int nr;
    float R[kMaxRadii];
    RampStep st[kMaxRadii];
    double smax;  // largest slopes of the two rows, added
};

double cumulative(const Table& t, bool back, double rho) {
    double c = 0.0, lo = 0.0;
    for (int q = 0; q < t.nr; q++) {
        const double sig = back ? t.st[q].sigb : t.st[q].sigf, hi = t.st[q].r;
        if (rho <= hi) return c + sig * (rho - lo);
        c += sig * (hi - lo);
        lo = hi;
    }
    return c;
}

// Both walks of destination j, sample by sample, in FP64.
double walk_direct(const RampLine& L, int j, const Table& t) {
    const double rlast = t.st[t.nr - 1].r, rprev = t.st[t.nr - 2].r;
    const bool exits = (double)L.cn - (double)L.c0 > rprev;
    double sum = 0.0;
    if (j > 0) {
        const double P = (double)L.c[j - 1] + (double)L.s[j - 1].x;
        double last = 0.0;
        for (int k = j - 1; k >= 0; k--) {
            if (exits && L.c[k] < (float)(P - rlast)) break;
            const double C = cumulative(t, true, P - (double)L.c[k]);
            sum += (C - last) * (double)L.s[k].y;
            last = C;
            if (exits && L.c[k] < (float)(P - rprev)) break;
        }
    }
    if (j < L.n - 1) {
        const double P = (double)L.c[j + 1] - (double)L.s[j + 1].x;
        double last = 0.0;
        for (int k = j + 1; k < L.n; k++) {
            if (exits && L.c[k] > (float)(P + rlast)) break;
            const double C = cumulative(t, false, (double)L.c[k] - P);
            sum += (C - last) * (double)L.s[k].y;
            last = C;
            if (exits && L.c[k] > (float)(P + rprev)) break;
        }
    }
    return sum;
}

}  // namespace

int main(int argc, char** argv) {
    const int nlines = argc > 1 ? std::atoi(argv[1]) : 1000;
    std::mt19937 rng(argc > 2 ? (unsigned)std::atoi(argv[2]) : 5u);
    std::uniform_real_distribution<float> U01(0.f, 1.f);
    const float radii[24] = {0.05f, 0.1f, 0.15f, 0.2f, 0.3f, 0.4f, 0.5f, 0.6f, 0.8f, 1.0f, 1.5f, 2.0f,
                             3.0f,  4.0f, 5.0f,  6.0f, 8.0f, 10.f, 15.f, 20.f, 30.f, 40.f, 50.f, 60.f};
    const float dens[5] = {1.0f, 0.25f, 1.85f, 0.001f, 0.f}, delr = 0.2f;
    uint64_t dests = 0, mismatch = 0, ended = 0, single = 0, late = 0;
    double worst = 0.0;
    std::string first;
    for (int li = 0; li < nlines; li++) {
        const bool behind = li & 1;
        const int n = li % 7 == 0 ? 1 + (int)(U01(rng) * 4.f) : 1 + (int)(U01(rng) * (li % 11 == 0 ? 1023.f : 300.f));
        Table t;
        t.nr = 2 + (int)(U01(rng) * 22.99f);  // (short tables end inside the line)
        t.smax = 0.0;
        double smax[2] = {0.0, 0.0};
        for (int q = 0; q < t.nr; q++) {
            t.R[q] = radii[q];
            const double lo = q ? (double)radii[q - 1] : 0.0, w = (double)radii[q] - lo;
            auto row = [](double r, double a, double b) { return a * (1.0 - std::exp(-r / b)); };
            t.st[q].r = (double)radii[q];
            t.st[q].sigf = (double)(float)((row(radii[q], 1.0, 1.7) - row(lo, 1.0, 1.7)) / w);
            t.st[q].sigb = (double)(float)((row(radii[q], 0.4, 0.9) - row(lo, 0.4, 0.9)) / w);
            t.st[q].pad = 0.0;
            smax[0] = std::max(smax[0], t.st[q].sigf);
            smax[1] = std::max(smax[1], t.st[q].sigb);
        }
        t.smax = smax[0] + smax[1];
        Fenced<float2> s((size_t)n, behind);
        Fenced<float> c((size_t)n + 4, behind);
        Fenced<double> E((size_t)n + 1, behind), E2((size_t)n + 1, behind);
        Fenced<uint16_t> lb(2 * (size_t)n + 4, behind);
        float T = 0.5f + U01(rng), tmax = 0.f;
        for (int k = 0; k < n;) {
            const int run = 1 + (int)(U01(rng) * 60.f), m = (int)(U01(rng) * 4.99f);
            const bool zero = U01(rng) < 0.15f;
            for (int q = 0; q < run && k < n; q++, k++) {
                T *= 0.97f + 0.02f * U01(rng);
                s.p[k] = make_float2(0.5f * (delr * dens[m]), zero ? 0.f : T);
                tmax = std::max(tmax, s.p[k].y);
            }
        }
        if (li % 5 == 0) s.p[0].x = std::pow(10.f, 1.f + 5.f * U01(rng));  // the first sample dwarfs the rest
        double P = 0.0, e1 = 0.0, e2 = 0.0;
        for (int k = 0; k < n; k++) {
            c.p[k] = (float)(P + (double)s.p[k].x);
            P += 2.0 * (double)s.p[k].x;
        }
        for (int q = 0; q < 4; q++) c.p[n + q] = INFINITY;
        for (int k = 0; k < n; k++) {
            const double tp = k > 0 ? (double)s.p[k - 1].y : 0.0, tn = k + 1 < n ? (double)s.p[k + 1].y : 0.0;
            E.p[k] = e1;
            E2.p[k] = e2;
            e1 = std::fma((double)s.p[k].y - tp, (double)c.p[k], e1);
            e2 = std::fma((double)s.p[k].y - tn, (double)c.p[k], e2);
        }
        E.p[n] = e1;
        E2.p[n] = e2;
        RampLine L;
        L.c = c.p;
        L.E = E.p;
        L.E2 = E2.p;
        L.s = s.p;
        L.lb = lb.p;
        L.n = n;
        L.U = 2 * n;
        L.c0 = c.p[0];
        L.cn = c.p[n - 1];
        L.invD = ramp_cells(L.c0, L.cn, L.U);
        const float D = L.invD > 0.f ? (L.cn - L.c0) / (float)L.U : 0.f;
        if (L.invD == 0.f) single++;
        int u = 0;
        for (int k = 0; k < n; k++)
            for (const int u1 = ramp_cell_after(L.c0, D, L.invD, L.U + 2, c.p[k]); u < u1; u++) lb.p[u] = (uint16_t)k;
        for (; u < L.U + 4; u++) lb.p[u] = (uint16_t)n;
        if ((double)L.cn - (double)L.c0 > t.st[t.nr - 2].r) ended++;
        const double tol = 2.0 * t.smax * (double)tmax * (double)(std::nextafter(L.cn, INFINITY) - L.cn) + 1e-12;
        for (int j = 0; j < n; j++) {
            uint32_t iters = 0;
            LateLane::left = (int)(rng() % 4 ? rng() % (uint32_t)(t.nr + 1) : 0);
            late += LateLane::left > 0;
            const double v = ramp_walk<true, true, LateLane>(L, j, t.st, t.nr, iters), w = walk_direct(L, j, t);
            const double err = std::fabs(v - w) / tol;
            worst = std::max(worst, err);
            if (!(err <= 1.0)) {
                if (!mismatch) {
                    char buf[200];
                    std::snprintf(buf, sizeof(buf), "line %d n %d nr %d j %d: %.12g against %.12g", li, n, t.nr, j, v, w);
                    first = buf;
                }
                mismatch++;
            }
            dests++;
        }
    }
    std::printf("{\"lines\": %d, \"destinations\": %" PRIu64 ", \"lines_beyond_the_radii\": %" PRIu64
                ", \"single_cell_lines\": %" PRIu64 ", \"late_lanes\": %" PRIu64 ", \"mismatch\": %" PRIu64
                ", \"worst_of_tolerance\": %.3f, \"first\": \"%s\"}\n",
                nlines, dests, ended, single, late, mismatch, worst, first.c_str());
    return mismatch ? 1 : 0;
}
