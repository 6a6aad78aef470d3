// A program over the C++ interface (include/ug_gpu/gpu_algebra.hpp) for what
// only that interface can do: settings changed between two uses of one object.
//   settings_client base_level   a matrix multigrid whose base level is lowered
//   settings_client precision    a multigrid whose precision is set after init,
//                                in a BiCGStab solve
// Prints what it compares; exit status 0 if every comparison holds.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <vector>

#include "ug_gpu/gpu_algebra.hpp"

using namespace ug::gpu;

namespace {

std::vector<double> values(const GPUVector& v) {
    std::vector<double> h((size_t)v.size());
    v.download(h.data());
    return h;
}

GPUVector vector_of(int64_t n, int seed) {
    std::vector<double> h((size_t)n);
    uint32_t s = 12345u + 977u * (uint32_t)seed;
    for (auto& x : h) {
        s = s * 1664525u + 1013904223u;
        x = (double)(s >> 8) / (1 << 24) - 0.5;
    }
    GPUVector v(n);
    v.upload(h.data());
    return v;
}

bool equal(const char* what, const GPUVector& a, const GPUVector& b) {
    const auto x = values(a), y = values(b);
    bool same = x.size() == y.size();
    for (size_t i = 0; same && i < x.size(); ++i) same = x[i] == y[i];
    double n2 = 0.0;
    for (double v : x) n2 += v * v;
    std::printf("%s: %s (norm %.6e)\n", what, same ? "equal" : "DIFFERENT", std::sqrt(n2));
    std::fflush(stdout);
    return same && n2 > 0.0 && std::isfinite(n2);
}

// the level matrices of a Q2 hierarchy
struct Q2Levels {
    std::vector<std::shared_ptr<GPUSparseMatrix>> A, P, R;
    explicit Q2Levels(int refs) {
        Q2Discretization q(refs);
        q.set_source(1.0);
        for (int l = 0; l <= refs; ++l) {
            for (auto* v : {&A, &P, &R}) v->push_back(std::make_shared<GPUSparseMatrix>());
            GPUVector b(q.num_dofs(l));
            q.assemble_linear(l, *A[l], b);
            if (l == 0) continue;
            q.prolongation(l, *P[l]);
            q.restriction(l, *P[l], *R[l]);
        }
    }
};

// one object: initialised and applied with the base level `high`, then with
// the base level `low`; the second correction is that of a new object
bool base_level(int refs, int high, int low) {
    Q2Levels q(refs);
    auto J = std::make_shared<MatrixOperator>(q.A[refs]);
    const int64_t n = q.A[refs]->num_rows();
    const GPUVector d = vector_of(n, refs);
    GPUVector c(n), ref(n);
    MatrixMultiGrid g;
    g.set_levels(q.A, q.P, q.R);
    for (int base : {high, low, high}) {
        g.set_base_level(base);
        if (!g.init(J) || !g.apply(c, d)) return false;
        MatrixMultiGrid fresh;
        fresh.set_levels(q.A, q.P, q.R);
        fresh.set_base_level(base);
        if (!fresh.init(J) || !fresh.apply(ref, d)) return false;
        char what[64];
        std::snprintf(what, sizeof(what), "refs %d base level %d", refs, base);
        if (!equal(what, c, ref)) return false;
    }
    // another base level without a new init is refused
    for (int base : {low, refs + 1, -1}) {
        g.set_base_level(base);
        bool refused = false;
        try {
            g.apply(c, d);
        } catch (const UGError&) {
            refused = true;
        }
        std::printf("base level %d without init: %s\n", base, refused ? "refused" : "ACCEPTED");
        if (!refused) return false;
    }
    return true;
}

// the precision set on the multigrid after init counts from the next init on:
// the solve in between is the one before it, the one behind it that of a new
// multigrid of that precision
bool precision(int refs, Precision from, Precision to) {
    auto disc = std::make_shared<DomainDiscretization>(2, refs);
    disc->set_velocity(20.0, 10.0, 5.0);
    auto A = std::make_shared<GPUSparseMatrix>();
    GPUVector b;
    disc->assemble_linear(*A, b);
    auto J = std::make_shared<MatrixOperator>(A);
    auto gmg = std::make_shared<AssembledMultiGridCycle>(disc);
    gmg->set_precision(from);
    BiCGStab S;
    S.set_preconditioner(gmg);
    if (!S.init(J)) return false;
    GPUVector x(b.size()), y(b.size());
    auto solve = [&](BiCGStab& s, GPUVector& v) {
        v.set(0.0);
        return s.apply(v, b);
    };
    if (!solve(S, x)) return false;
    gmg->set_precision(to);
    if (gmg->precision() != from || !solve(S, y) || !equal("precision set, no init", x, y)) return false;
    if (!S.init(J) || gmg->precision() != to || !solve(S, y)) return false;
    auto fresh = std::make_shared<AssembledMultiGridCycle>(disc);
    fresh->set_precision(to);
    BiCGStab F;
    F.set_preconditioner(fresh);
    return F.init(J) && solve(F, x) && equal("precision after init", x, y);
}

}  // namespace

int main(int argc, char** argv) {
    bool ok = false;
    try {
        if (argc > 1 && !std::strcmp(argv[1], "base_level")) ok = base_level(2, 1, 0) && base_level(3, 2, 0);
        if (argc > 1 && !std::strcmp(argv[1], "precision"))
            ok = precision(1, Precision::F32, Precision::F64) && precision(2, Precision::F64, Precision::F32);
    } catch (const std::exception& e) {
        std::printf("error: %s\n", e.what());
    }
    return ok ? 0 : 1;
}
