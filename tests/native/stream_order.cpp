// Programs against the host classes on the runtime of fake_hip.cpp: what is queued, waited for and refused.
// One scenario per run, named by the argument; exit status 0 when it holds.
#include <cstdio>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include "../../include/grape_hip.h"
#include "../../grape_amd/host/hyrax.hpp"
#include "../../grape_amd/host/prove.hpp"
#include "../../grape_amd/host/tlookup.hpp"

extern "C" {
unsigned long fake_pending(const void* stream);
unsigned long fake_unjoined();
unsigned long fake_launches();
unsigned long fake_copies();
void fake_queue(const void* stream);
}

static int failures = 0;
static void expect(bool ok, const char* what) {
    if (!ok) {
        std::printf("does not hold: %s\n", what);
        failures++;
    }
}
static affine_t* device_points(size_t n) {
    void* p = nullptr;
    grape_host::ensure_init();
    grape_host::check(grape_malloc(&p, sizeof(affine_t) * n), "grape_malloc");
    return static_cast<affine_t*>(p);
}

// A range lookup whose proof is refused between its long rounds and its commitments (com_m has fewer rows than layers): the
// long rounds' sums are being finished on a stream of their own then, and everything they use is given back.
static void refused_lookup() {
    const uint D = 1u << 18, cols = 64, len = 256, layers = 64;
    bn128 G = bn128::one();
    Hyrax hyrax(layers, cols, device_points(256 * cols), G, 1);
    tLookupRange lookup(-128, len);
    FrTensor S(D), A(D);
    int* ints = reinterpret_cast<int*>(device_points(D / 16));
    double seconds = 0;
    std::string error;
    try {
        lookup.prove(ints, S, A, random_vec(18), hyrax, cols, seconds);
    } catch (const std::exception& e) {
        error = e.what();
    }
    expect(error.find("Size too small") == 0, "the commitment of the multiplicities is refused");
    expect(fake_unjoined() == 0, "no stream is left with work that nothing waits for");
}

int main(int argc, char** argv) {
    const std::map<std::string, std::function<void()>> scenarios = {
        {"refused_lookup", refused_lookup},
    };
    auto it = scenarios.find(argc > 1 ? argv[1] : "");
    if (it == scenarios.end()) return 2;
    try {
        it->second();
    } catch (const std::exception& e) {
        std::printf("%s\n", e.what());
        return 1;
    }
    return failures ? 1 : 0;
}
