// The band solver (band.hip, host code and kernels) on the host HIP runtime of
// host_hip/, on random symmetric matrices of n equations and half-bandwidth b
// with one slot per joint.
//   band_host solve n b [xcds slots]   fused and split factors bitwise equal, each
//                                      sweep schedule solves the system, FP64 and FP32
//   band_host pair n b xcds slots [counted]  two handles at once: their factorizations
//                                      and solves, each the result of a handle alone
//   band_host unfactored               a solve without a factor is an error
//   band_host memory                   a factorization whose k-th allocation fails,
//                                      for every k, is an error and can be repeated
// Prints what it finds and returns 1 on the first thing that is wrong.
#include "../cu-bens_amd/csrc/band.hip"

#include <cstdio>

using cb::BandLDLT;
using cb::Dev;

struct Problem {
    Dev d;
    long n, b;
    std::vector<double> A;   // dense
    Problem(long n_, long b_, uint64_t seed = 1) : n(n_), b(std::min(b_, n_ - 1)), A(size_t(n_ * n_), 0.0) {
        uint64_t state = seed;
        auto rnd = [&] {
            state = state * 6364136223846793005ull + 1442695040888963407ull;
            return double(state >> 11) / 9007199254740992.0 - 0.5;
        };
        std::vector<int32_t> rp(1, 0), ci, eq;
        std::vector<double> K;
        for (long i = 0; i < n; ++i)
            for (long j = std::max(0L, i - b); j <= i; ++j)
                A[size_t(i * n + j)] = A[size_t(j * n + i)] = i == j ? 0.3 * double(b) + 1.0 : rnd();
        for (long i = 0; i < n; ++i) {
            for (long j = std::max(0L, i - b); j <= std::min(n - 1, i + b); ++j) {
                ci.push_back(int32_t(j));
                K.push_back(A[size_t(i * n + j)]);
            }
            rp.push_back(int32_t(ci.size()));
            eq.push_back(int32_t(i));
        }
        d.nj = d.nslot = n;
        d.bs = 1;
        up(d.rowptr, rp);
        up(d.colidx, ci);
        up(d.eq_of_slot, eq);
        up(d.K, K);
    }
    template <class P, class V> static void up(P*& dst, const V& v) {
        dst = cb::dalloc<P>(v.size());
        cb::h2d(dst, v.data(), v.size(), nullptr);
    }
    // largest residual of a solve, over the sizes of its terms
    template <class R> double solve(BandLDLT<R>& f) const {
        std::vector<double> rhs, x(static_cast<size_t>(n));
        for (long i = 0; i < n; ++i) rhs.push_back(double((i * 37) % 101) / 50.0 - 1.0);
        double *db = nullptr, *dx = cb::dalloc<double>(x.size());
        up(db, rhs);
        f.solve(db, dx);
        cb::d2h(x.data(), dx, x.size(), nullptr);
        double worst = 0, xm = 0, am = 0;
        for (double v : x) xm = std::max(xm, std::fabs(v));
        for (long i = 0; i < n; ++i) {
            double r = -rhs[size_t(i)], a = 0;
            for (long j = 0; j < n; ++j) {
                r += A[size_t(i * n + j)] * x[size_t(j)];
                a += std::fabs(A[size_t(i * n + j)]);
            }
            worst = std::max(worst, std::fabs(r));
            am = std::max(am, a);
        }
        return worst / (am * xm + 1.0);
    }
};

template <class R> bool same(const R* a, const R* b, size_t n) { return std::memcmp(a, b, n * sizeof(R)) == 0; }

template <class R> int solve_all(long n, long b, double eps) {
    Problem p(n, b);
    BandLDLT<R> split, f;
    split.setup(n, b, nullptr);
    split.split = true;
    f.setup(n, b, nullptr);
    if (split.factor(p.d) != 0) return std::printf("split schedule: not factored\n"), 1;
    std::printf("%ld equations, %ld tile rows, %d tiles below the diagonal\n", n, f.nt, f.w);
    for (int sweeps = 0; sweeps < 3; ++sweeps) {
        f.chained = sweeps != 1;
        f.blocks = sweeps == 2;
        if (f.factor(p.d) != 0) return std::printf("fused schedule: not factored\n"), 1;
        for (long I = 0; I < f.nt; ++I) {
            bool ok = same(f.linv + I * cb::TT, split.linv + I * cb::TT, cb::TT) &&
                      same(f.piv + I * cb::T, split.piv + I * cb::T, cb::T);
            for (long J = std::max(0L, I - f.w); J < I; ++J) {
                const long t = cb::tile_index(I, J, f.w) * cb::TT;
                ok = ok && same(f.tiles + t, split.tiles + t, cb::TT) && same(f.tiles_t + t, split.tiles_t + t, cb::TT);
            }
            if (!ok) return std::printf("tile row %ld: fused and split factors differ\n", I), 1;
        }
        const double eta = p.solve(f);
        std::printf("sweeps %d: backward error %.2e\n", sweeps, eta);
        if (!(eta < eps)) return 1;
    }
    return 0;
}

// Two handles' launches, the i-th of one beside the i-th of the other
template <class F> void side_by_side(F&& a, F&& b) {
    std::vector<host_hip::Launch> la, lb;
    host_hip::held = &la;
    a();
    host_hip::held = &lb;
    b();
    host_hip::held = nullptr;
    for (size_t i = 0; i < la.size(); ++i) host_hip::run({la[i], lb[i]});
}

int pair(long n, long b, int xcds, int slots, int counted) {
    Problem p(n, b);
    BandLDLT<double> alone, two[2];
    for (int sweeps = 0; sweeps < 3; ++sweeps) {
        auto prepare = [&](BandLDLT<double>& f) {
            f.setup(n, b, nullptr);
            f.chained = sweeps != 1;
            f.blocks = sweeps == 2;
            f.spin_limit = 200000;
            f.counted = counted;
        };
        for (BandLDLT<double>* f : {&alone, &two[0], &two[1]}) prepare(*f);
        host_hip::xcds = 4;
        host_hip::slots = 2;
        if (alone.factor(p.d) != 0 || !(p.solve(alone) < 1e-14)) return 1;
        std::vector<double> x(static_cast<size_t>(n), 1.0);
        double *rhs = nullptr, *out = cb::dalloc<double>(x.size());
        Problem::up(rhs, x);
        alone.solve(rhs, out);
        host_hip::xcds = xcds;
        host_hip::slots = slots;
        auto factor = [&](int i) { return [&, i] { two[i].factor(p.d); }; };
        auto solve = [&](int i) { return [&, i] { two[i].solve(rhs, out); }; };
        side_by_side<std::function<void()>>(factor(0), factor(1));
        const int bad = two[0].flag[0] | two[1].flag[0];
        std::printf("sweeps %d: factorizations %s\n", sweeps, bad ? "stopped at a wait's bound" : "ended");
        if (bad) return 1;
        side_by_side<std::function<void()>>(solve(0), solve(1));
        const int bad2 = two[0].flag[0] | two[1].flag[0];
        std::printf("sweeps %d: solves %s\n", sweeps, bad2 ? "stopped at a wait's bound" : "ended");
        if (bad2) return 1;
        for (BandLDLT<double>& f : two)
            if (!same(f.piv, alone.piv, size_t(n)) || !same(f.xw, alone.xw, size_t(n)))
                return std::printf("the results differ from a handle's alone\n"), 1;
    }
    return 0;
}

template <class F> bool refused(F&& call) {
    try {
        call();
    } catch (const cb::DeviceError& e) {
        std::printf("refused: %s\n", e.msg.c_str());
        return true;
    }
    std::printf("not refused\n");
    return false;
}

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    auto arg = [&](int i, long other) { return argc > i ? std::atol(argv[i]) : other; };
    if (what == "solve") {
        const long n = arg(2, 200), b = arg(3, 70);
        host_hip::xcds = int(arg(4, 4));
        host_hip::slots = int(arg(5, 2));
        // 64-term sums of products, a few hundred of them after one another
        return solve_all<double>(n, b, 1e-14) || solve_all<float>(n, b, 1e-6);
    }
    if (what == "pair") return pair(arg(2, 600), arg(3, 200), int(arg(4, 4)), int(arg(5, 2)), int(arg(6, 1024)));
    if (what == "unfactored") {
        Problem p(400, 70);
        for (int sweeps = 0; sweeps < 3; ++sweeps) {
            BandLDLT<double> f;
            f.chained = sweeps != 1;
            f.blocks = sweeps == 2;
            f.setup(p.n, p.b, nullptr);
            if (!refused([&] { p.solve(f); })) return 1;
            if (f.factor(p.d) != 0 || !(p.solve(f) < 1e-14)) return 1;
            f.setup(p.n, p.b, nullptr);   // the new handle has no factor either
            if (!refused([&] { p.solve(f); })) return 1;
        }
        return 0;
    }
    if (what == "memory") {
        Problem p(400, 70);
        for (bool blocks : {false, true}) {
            int failures = 0;
            for (long k = 0;; ++k) {
                BandLDLT<double> f;
                f.blocks = blocks;
                f.setup(p.n, p.b, nullptr);
                host_hip::fail_at = k;
                const bool failed = [&] {
                    try {
                        f.factor(p.d);
                        return false;
                    } catch (const cb::DeviceError&) {
                        return true;
                    }
                }();
                host_hip::fail_at = -1;
                if (!failed) break;
                ++failures;
                if (!refused([&] { p.solve(f); })) return 1;
                if (f.factor(p.d) != 0 || !(p.solve(f) < 1e-14)) return 1;
            }
            std::printf("%s sweeps: %d allocations, each failed once\n", blocks ? "block" : "chain", failures);
            if (!failures) return 1;
        }
        return 0;
    }
    return std::printf("what?\n"), 2;
}
