// The intervals of the Rys fits, in double and in float, at and next to every interval's ends up to the
// large-T limit: index inside the table, local variable in [-1, 1] up to rounding, both overloads on the same
// polynomial, and the float nodes and weights near the double ones.  Built and run by tests/test_host_rys.py.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <vector>

#include "../../iqcp_amd/csrc/rys.h"

using namespace qcg;

template <int N>
void check() {
    const double tmax = qcg_rys_tmax[N], T0 = 1 << qcg_rys_log2t0[N];
    std::vector<float> tabf(rys_tab_size<N>());
    for (int i = 0; i < rys_tab_size<N>(); ++i) tabf[i] = (float)qcg_rys_coef[qcg_rys_off[N] + i];
    std::vector<float> at;
    double lo = T0;
    for (int k = 0; k < qcg_rys_nint[N]; ++k) {
        const double h = std::ldexp(1.0, (int)std::floor(std::log2(lo)) - qcg_rys_bits[N]);
        for (double f : {0.0, 0.25, 0.5, 0.75, 1.0}) {
            const float t = (float)(lo - T0 + f * h);
            for (float v : {std::nextafter(t, -1.f), t, std::nextafter(t, 1e9f)})
                if (v >= 0.f && v < (float)tmax) at.push_back(v);
        }
        lo += h;
    }
    at.push_back(std::nextafter((float)tmax, 0.f));
    int bad = 0, split = 0;
    double smax = 0.0, err = 0.0;
    for (float t : at) {
        float sf;
        double sd;
        const int kf = rys_interval<N>(t, sf), kd = rys_interval<N>((double)t, sd);
        bad += kf < 0 || kf >= qcg_rys_nint[N] || kd < 0 || kd >= qcg_rys_nint[N] || std::abs(kf - kd) > 1;
        split += kf != kd;
        smax = std::max({smax, std::fabs((double)sf), std::fabs(sd)});
        float xf[N], wf[N];
        double xd[N], wd[N];
        rys_eval_tab<float, N>(t, tabf.data(), xf, wf);
        rys_eval_tab<double, N>((double)t, qcg_rys_coef + qcg_rys_off[N], xd, wd);
        for (int i = 0; i < N; ++i) err = std::max({err, std::fabs(xf[i] / xd[i] - 1.0), std::fabs(wf[i] / wd[i] - 1.0)});
    }
    std::printf("points_%d %zu\nbad_%d %d\nsplit_%d %d\nsmax_%d %.9f\nerr32_%d %.3e\n", N, at.size(), N, bad, N, split, N, smax, N, err);
}

int main() {
    check<1>(), check<2>(), check<3>(), check<4>(), check<5>(), check<6>(), check<7>();
    return 0;
}
