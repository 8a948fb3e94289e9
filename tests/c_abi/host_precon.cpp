// A C++ host of libpar-ilu0-gmres.so that solves with its own preconditioner
// (the diagonal) through SetPreconditioner and reads the true residual right
// after the solve, on systems of 40^2 rows (one workgroup per Gram-Schmidt step)
// and 100^2 (the whole GPU).  Prints "residual <device> <host>" for each; exit
// status 0 when both converge.
#include <cmath>
#include <cstdio>
#include <vector>

#include "gmres.hpp"

namespace {

double residual(const CsrMatrix* a, const std::vector<double>& b, std::vector<double>& x) {
    std::vector<double> ax(b.size());
    CsrMatVec(const_cast<CsrMatrix*>(a), x.data(), ax.data());
    double s = 0.0;
    for (size_t i = 0; i < b.size(); ++i) s += (b[i] - ax[i]) * (b[i] - ax[i]);
    return std::sqrt(s);
}

bool solve(int side) {
    const int n = side * side;
    std::vector<int> rp(1, 0), ci;
    for (int i = 0; i < n; ++i) {
        const int x = i % side;
        if (i >= side) ci.push_back(i - side);
        if (x > 0) ci.push_back(i - 1);
        ci.push_back(i);
        if (x + 1 < side) ci.push_back(i + 1);
        if (i + side < n) ci.push_back(i + side);
        rp.push_back(static_cast<int>(ci.size()));
    }
    CsrMatrix a = CSR_MATRIX_DEFAULT;
    SetupCsrMatrix(&a, n, static_cast<int>(ci.size()));
    std::vector<double> diag(n), b(n), x(n, 0.0);
    for (int i = 0; i <= n; ++i) a.row_ptr[i] = rp[i];
    for (int i = 0; i < n; ++i) {
        diag[i] = 5.0 + i % 7;
        b[i] = 1.0 + i % 3;
        for (int k = rp[i]; k < rp[i + 1]; ++k) {
            a.col_idx[k] = ci[k];
            a.value[k] = ci[k] == i ? diag[i] : -1.0;
        }
    }
    bool ok;
    double got;
    {
        lljbash::PreconditionedGmres g;
        g.SetPreconditioner([&](const double* v, double* z) {
            for (int i = 0; i < n; ++i) z[i] = v[i] / diag[i];
        });
        ok = g.Solve(&a, b.data(), x.data()).first;
        got = g.LastTrueResidual();
    }
    std::printf("residual %.17g %.17g\n", got, residual(&a, b, x));
    DestroyCsrMatrix(&a);
    return ok;
}

}  // namespace

int main() {
    const bool small = solve(40), large = solve(100);
    return small && large ? 0 : 2;
}
