// Host side of the parametric potential model (sld_model.h): the forms of
// DD05.cpp:6-164 and JijFe.cpp:5-43 with their coefficients taken from the
// parameter vector, sampled like potential_CPU.cpp:61-170 (10^6 points, the
// 6-point central-difference derivative) by the device (sld_model_tab.hip).
// Every parameter except the exchange cutoff rc enters a table linearly, so
// the derivative of a table with respect to it is the table of its basis
// function, built the same way; the rc derivative is the table of dJ/drc at
// the current parameters.
//
// The pair term's quintic bridge (1.8 < r <= 2 A) is evaluated as the bridge
// of the ZBL end alone plus sum_k V_k times the bridge of knot k alone. This
// is the same polynomial as DD05.cpp:88-158's single closed form (the bridge
// is linear in its six end values), but the closed form cancels large terms
// and carries rounding noise of about 1e-9 of V (1e-7 of V' after the
// 6-point derivative) that varies with V; split, the noise sits in the
// V-independent ZBL part and the model is smooth in V_k. The nine
// polynomials' values do not depend on theta and are made here once.
#include <algorithm>
#include <cmath>
#include <mutex>
#include <thread>
#include <utility>
#include <vector>

#include "sld_common.h"
#include "sld_model.h"
#include "sld_tables.h"
#include "sld_threads.h"

namespace sld {
namespace {

// knots of the density and pair splines (DD05.cpp:26-37,70-85), as in sld_model_device.h
const double kFR[6] = {3.0, 2.8666666666666666, 2.7333333333333333, 2.6, 2.4, 2.3};
const double kVR[8] = {4.1, 3.8, 3.5, 3.2, 2.9, 2.6, 2.4, 2.3};

double quintic(const Bridge& b, double r) {
    using std::pow;
    const double* a = b.a;
    return a[5] * pow(r, 5) + a[4] * pow(r, 4) + a[3] * pow(r, 3) + a[2] * pow(r, 2) + a[1] * r + a[0];
}

void bridge_polynomials(Bridge (&q)[9]) {
    const double x2 = 2.0;
    q[0] = bridge_from_ends(zbl_ends(), 0e0, 0e0, 0e0);
    const ZblEnds zero = {0e0, 0e0, 0e0};
    for (int k = 0; k < 8; ++k) {
        double g = 0e0, dg = 0e0, d2g = 0e0;
        if (x2 < kVR[k]) {
            g = std::pow(kVR[k] - x2, 3);
            dg = -3e0 * std::pow(kVR[k] - x2, 2);
            d2g = 6e0 * (kVR[k] - x2);
        }
        q[1 + k] = bridge_from_ends(zero, g, dg, d2g);
    }
}

// the r of table entry n, as the device computes it
double entry_r(double rmax, int n) { return rmax / (double)kNInput * (double)(n + 1); }

void fill_bridge(double rmax, ModelBridge& t) {
    Bridge q[9];
    bridge_polynomials(q);
    // rows whose stencil (x +- 3x/1000) can reach (1.8, 2.0], with a margin
    const double per = kNInput / rmax;
    t.row0 = std::max(0, std::min(kNInput, (int)(1.8 / 1.003 * per) - 4));
    t.nrow = std::max(0, std::min(kNInput, (int)(2.0 / 0.997 * per) + 4) - t.row0);
    t.q.assign((size_t)std::max(t.nrow, 1) * kModelBridgeRow, 0.0);
    auto work = [&](int a, int b) {
        for (int k = a; k < b; ++k) {
            const double r = entry_r(rmax, t.row0 + k);
            const double dx = r / 1000e0;
            const double x[7] = {r, r + dx, r - dx, r + 2 * dx, r - 2 * dx, r + 3 * dx, r - 3 * dx};
            for (int s = 0; s < 7; ++s)
                if (x[s] > 1.8 && x[s] <= 2.0)
                    for (int p = 0; p < 9; ++p) t.q[((size_t)k * 7 + s) * 9 + p] = quintic(q[p], x[s]);
        }
    };
    const int nt = (int)std::min(std::max(std::thread::hardware_concurrency(), 1u), 16u);
    const int chunk = (t.nrow + nt - 1) / nt;
    run_parts(nt, [&](int k) { work(k * chunk, std::min((k + 1) * chunk, t.nrow)); });
}

}  // namespace

std::shared_ptr<const ModelBridge> model_bridge(double rcut_max) {
    static std::mutex mu;
    static std::vector<std::pair<double, std::shared_ptr<const ModelBridge>>> cache;  // the last used first
    std::lock_guard<std::mutex> lock(mu);
    auto it = std::find_if(cache.begin(), cache.end(), [&](const auto& e) { return e.first == rcut_max; });
    if (it == cache.end()) {
        auto t = std::make_shared<ModelBridge>();
        fill_bridge(rcut_max, *t);
        if ((int)cache.size() == kModelBridges) cache.pop_back();
        it = cache.emplace(cache.end(), rcut_max, std::move(t));
    }
    std::rotate(cache.begin(), it, it + 1);
    return cache.front().second;
}

void model_default_params(double* th) {
    const double a[6] = {0.9332056681088162, -1.162558782567700, -0.3502026949249225,
                         0.4287820835430028, 4.907925057809273,  -5.307049068415304};
    const double V[8] = {-0.1960674387419232, 0.3687525935422963, -1.505333614924853, 4.948907078156191,
                         -4.894613262753399,  3.468897724782442,  -1.792218099820337, 80.22069592246987};
    for (int k = 0; k < 6; ++k) th[P_A0 + k] = a[k];
    for (int k = 0; k < 8; ++k) th[P_V0 + k] = V[k];
    th[P_AA] = 4.100199340884814;
    th[P_BB] = 1.565647547483517;
    th[P_JA] = 0.870;
    th[P_JRC] = 3.75;
    th[P_LA + 0] = -0.744824;
    th[P_LA + 1] = 0.345295;
    th[P_LA + 2] = -0.00790205;
    th[P_LA + 3] = 0e0;
}

ModelCoef model_coef(const double* th, double rcut_max, const ModelBridge& bridge) {
    ModelCoef m;
    for (int k = 0; k < 6; ++k) m.a[k] = th[P_A0 + k];
    for (int k = 0; k < 8; ++k) m.V[k] = th[P_V0 + k];
    m.aa = th[P_AA];
    m.bb = th[P_BB];
    m.JA = th[P_JA];
    m.Jrc = th[P_JRC];
    m.as = 0.88535e0 * 0.52917720859e0 / (2e0 * std::pow(26e0, 0.23));  // DD05.cpp:45-62
    m.ln2 = std::log(2e0);
    double f1 = 0e0;
    for (int i = 0; i < 6; ++i) f1 += m.a[i] * std::pow(kFR[i] - 1e0, 3);
    m.rmax = rcut_max;
    m.rhomax = 2e0 * f1 < 1000e0 ? 1000e0 : 2e0 * f1;
    m.row0 = bridge.row0;
    return m;
}

}  // namespace sld
