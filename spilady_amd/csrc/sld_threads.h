// Host loops in parts on several threads.
#pragma once

#include <exception>
#include <thread>
#include <vector>

namespace sld {

// part(0) .. part(nt - 1), each on a thread of its own where one can be had; the
// calling thread does the last part and all that got no thread. What a part
// throws is thrown here, once every part has ended.
template <class F>
void run_parts(int nt, F part) {
    std::vector<std::exception_ptr> thrown(nt);
    auto run = [&](int k) {
        try {
            part(k);
        } catch (...) {
            thrown[k] = std::current_exception();
        }
    };
    std::vector<std::thread> th;
    th.reserve(nt);
    int k = 0;
    try {
        for (; k + 1 < nt; ++k) th.emplace_back(run, k);
    } catch (...) {
        // no thread to be had
    }
    for (; k < nt; ++k) run(k);
    for (auto& x : th) x.join();
    for (auto& e : thrown)
        if (e) std::rethrow_exception(e);
}

}  // namespace sld
