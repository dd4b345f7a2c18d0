// The field products of grape_amd/csrc/fp30.hpp and fr26.hpp on limbs as they are, so that the CPU test-suite can put
// operands at the bounds of their columns.
#include <cstring>
#include "../../grape_amd/csrc/fp30.hpp"
#include "../../grape_amd/csrc/fr26.hpp"
using namespace grape;

static Fp30 load(const int32_t* p) {
    Fp30 a;
    memcpy(a.v, p, sizeof a.v);
    return a;
}
extern "C" {
int fp30_limbs() { return fp30::N; }
// a, b lazy or balanced as the function asks; s, u balanced; out: limbs
void fp30_apply(int op, const int32_t* a, const int32_t* b, const int32_t* s, const int32_t* u, int32_t* out) {
    const Fp30 A = load(a), B = load(b), S = load(s), U = load(u);
    Fp30 r;
    switch (op) {
    case 0: r = fp30::mul(A, B); break;
    case 1: r = fp30::mulb(A, B); break;
    case 2: r = fp30::mulb_below_p(A, B); break;
    case 3: r = fp30::mulb_less(A, B, S); break;
    case 4: r = fp30::mul_sub(A, B, S, U); break;
    case 5: r = fp30::sqr(A); break;
    case 6: r = fp30::sqr_below_p(A); break;
    case 7: r = fp30::sqr_less(A, S, U); break;
    case 8: r = fp30::balance(A); break;
    case 9: r = fp30::normalize(A); break;
    case 11: r = fp30::balance<true>(A); break;
    case 10: r = fp30::canonical(fp30::mul(A, B)); break;
    default: r = fp30::zero();
    }
    memcpy(out, r.v, sizeof r.v);
}
void fr26_product(const int32_t* a, const int32_t* b, int add_r, int32_t* out) {
    fr26::Limbs A, B;
    memcpy(A.v, a, sizeof A.v);
    memcpy(B.v, b, sizeof B.v);
    const fr26::Limbs r = fr26::product(A, B, add_r);
    memcpy(out, r.v, sizeof r.v);
}
void fr26_limb_sum(const int32_t* sum, int add_r, uint32_t* out) {
    fr26::Limbs s;
    memcpy(s.v, sum, sizeof s.v);
    const Fr r = fr26::limb_sum_to_fr(s, add_r);
    memcpy(out, r.v, sizeof r.v);
}
int fp30_zero(const int32_t* a, const int32_t* b) { return fp30::is_zero(fp30::mulb_below_p(load(a), load(b))) ? 1 : 0; }
}
