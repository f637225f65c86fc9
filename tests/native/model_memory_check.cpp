// sld_model_set_params on a device that refuses its k-th allocation, for every
// k: the call returns an error, and the next one starts anew and gives what an
// undisturbed context gives.
//   model_memory_check state   natom, sld_params, then r, p and s ([natom][3])
#include "spilady_hip.h"

#include <dlfcn.h>

#include <cstddef>
#include <cstdio>
#include <vector>

static int refuse_at = -1, count = 0;

extern "C" int hipMalloc(void** p, std::size_t n) {
    using Fn = int (*)(void**, std::size_t);
    static const Fn real = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "hipMalloc"));
    return count++ == refuse_at ? 2 /* hipErrorOutOfMemory */ : real(p, n);
}

int main(int, char** argv) {
    FILE* f = std::fopen(argv[1], "rb");
    int natom = 0;
    sld_params prm;
    if (!f || std::fread(&natom, sizeof(natom), 1, f) != 1 || std::fread(&prm, sizeof(prm), 1, f) != 1) return 1;
    std::vector<double> v(9 * (std::size_t)natom);
    if (std::fread(v.data(), sizeof(double), v.size(), f) != v.size()) return 1;
    std::fclose(f);
    sld_atoms at = {};
    at.r = v.data();
    at.p = v.data() + 3 * natom;
    at.s = v.data() + 6 * natom;
    double theta[64], want = 0.0;
    if (sld_model_default_params(theta)) return 1;
    int refused = 0;
    for (int k = -1;; ++k) {
        sld_ctx* c = nullptr;
        if (sld_create(&prm, &at, 0, &c)) {
            std::printf("create: %s\n", sld_last_error(c));
            return 1;
        }
        count = 0;
        refuse_at = k;
        const int rc = sld_model_set_params(c, theta);
        const bool hit = k >= 0 && count > k;
        refuse_at = -1;
        if (hit != (rc != 0)) return 2;
        if (hit) {
            ++refused;
            if (sld_model_set_params(c, theta)) {
                std::printf("second call after %d: %s\n", k, sld_last_error(c));
                return 3;
            }
        }
        double e = 0.0;
        if (sld_model_eval(c, &e, nullptr, nullptr)) return 4;
        if (k < 0) want = e;
        if (e != want) return 5;
        sld_destroy(c);
        std::printf("allocation %d %s\n", k, hit ? "refused" : "granted");
        std::fflush(stdout);
        if (k >= 0 && !hit) break;
    }
    std::printf("refused %d\n", refused);
    return refused > 10 ? 0 : 6;
}
