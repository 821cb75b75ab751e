// The learned preconditioner's kernels on the host HIP runtime of host_hip/,
// over the joint graph of an n x n triangulated panel: features, network,
// preconditioner, and loss and gradient of `pairs` vector pairs under one
// objective, or under each.  Prints the losses and the gradient's norms; an access past the end
// of a buffer ends the process with a segmentation fault.
#include "../cu-bens_amd/csrc/learned.hip"

#include <cstdio>

namespace cb {
namespace {
thread_local bf16_t sB[160 * 1024 / sizeof(bf16_t)];   // k_gemm's dynamic LDS
}
void bsr_spmv(Dev& d, const double* x, double* y) {
    for (long j = 0; j < d.nj; ++j)
        for (int p = 0; p < 6; ++p) {
            double s = 0;
            for (int32_t k = d.rowptr[j]; k < d.rowptr[j + 1]; ++k)
                for (int q = 0; q < 6; ++q) s += d.K[long(k) * 36 + p * 6 + q] * x[long(d.colidx[k]) * 6 + q];
            y[j * 6 + p] = s;
        }
}
}  // namespace cb

int main(int argc, char** argv) {
    const int n = argc > 1 ? std::atoi(argv[1]) : 3, pairs = argc > 2 ? std::atoi(argv[2]) : 2, m = n + 1;
    uint64_t state = 1;
    auto rnd = [&] {
        state = state * 6364136223846793005ull + 1442695040888963407ull;
        return double(state >> 11) / 9007199254740992.0 - 0.5;
    };
    cb::Dev d;
    d.uid = 1;
    d.nj = long(m) * m;
    d.nslot = d.nj * 6;
    std::vector<int32_t> rp(1, 0), ci, db, eq;
    std::vector<double> K;
    int32_t free_ = 0;
    for (int r = 0; r < m; ++r)
        for (int c = 0; c < m; ++c) {
            const int step[7][2] = {{-1, -1}, {-1, 0}, {0, -1}, {0, 0}, {0, 1}, {1, 0}, {1, 1}};
            for (auto& s : step) {
                const int rr = r + s[0], cc = c + s[1];
                if (rr < 0 || rr >= m || cc < 0 || cc >= m) continue;
                const bool diag = rr == r && cc == c;
                if (diag) db.push_back(int32_t(ci.size()));
                ci.push_back(rr * m + cc);
                for (int p = 0; p < 36; ++p) K.push_back(diag ? (p % 7 == 0 ? 8.0 : 0.0) : -0.2 * (p % 7 == 0));
            }
            rp.push_back(int32_t(ci.size()));
            for (int p = 0; p < 6; ++p) eq.push_back(r == 0 && p < 3 ? -1 : free_++);
        }
    d.nnzb = long(ci.size());
    auto up = [](auto*& dst, const auto& v) {
        dst = cb::dalloc<std::remove_reference_t<decltype(*dst)>>(v.size());
        cb::h2d(dst, v.data(), v.size(), nullptr);
    };
    up(d.rowptr, rp);
    up(d.colidx, ci);
    up(d.diagblk, db);
    up(d.eq_of_slot, eq);
    up(d.K, K);
    cb::Learned net(3);
    std::vector<float> p(size_t(net.nparams()));
    net.get_params(p.data());
    for (float& v : p)
        if (v == 0.f) v = float(0.04 * rnd());
    net.set_params(p.data());
    std::vector<const double*> r, u;
    for (int b = 0; b < pairs; ++b) {
        std::vector<double> x(size_t(d.nslot)), y;
        for (size_t i = 0; i < x.size(); ++i) x[i] = eq[i] >= 0 ? rnd() : 0.0;
        double *ud = nullptr, *rd = nullptr;
        up(ud, x);
        rd = cb::dalloc<double>(x.size());
        cb::bsr_spmv(d, ud, rd);
        r.push_back(rd);
        u.push_back(ud);
    }
    const int only = argc > 3 ? std::atoi(argv[3]) : -1;
    for (int objective = 0; objective < 3; ++objective) {
        if (only >= 0 && objective != only) continue;
        net.set_objective(objective);
        net.setup(d);
        const double loss = net.loss_grad(d, r.data(), u.data(), pairs);
        std::vector<float> g(p.size());
        net.get_grad(g.data());
        double s = 0;
        for (float v : g) s += double(v) * v;
        net.adam_step(1e-3f);
        double* z = cb::dalloc<double>(size_t(d.nslot));
        net.apply(d, r[0], z);
        std::printf("%ld joints %ld edges objective %d loss %.6e gradient %.6e\n", net.nv(), net.ne(), objective, loss,
                    std::sqrt(s));
        if (!std::isfinite(loss) || !std::isfinite(s) || !(s > 0)) return 1;
    }
    return 0;
}
