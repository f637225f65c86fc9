// The bridge polynomials that stay with the process: those of the last
// kModelBridges cutoffs, and one that is used again is not made again.
#include "sld_model.h"

#include <cstdio>

using namespace sld;

int main() {
    std::vector<std::weak_ptr<const ModelBridge>> seen;
    for (int k = 0; k < kModelBridges + 3; ++k) {
        const auto a = model_bridge(4.0 + 0.1 * k);
        seen.push_back(a);
        if (!seen.front().expired()) (void)model_bridge(4.0);  // keeps the first in use
        if (a->nrow <= 0 || a != model_bridge(4.0 + 0.1 * k)) return 1;
    }
    int alive = 0;
    for (const auto& w : seen) alive += !w.expired();
    std::printf("alive %d first %d last %d\n", alive, !seen.front().expired(), !seen.back().expired());
    return 0;
}
