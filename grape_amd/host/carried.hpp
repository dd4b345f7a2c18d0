// The host's side of the rounds that carry their weights (grape_carried_queue): the factors between a round's two sums and its
// polynomial, the ratios the carried tensor is folded by, and what is left in it in the end.  A round binds u_j and v_k
// (the last coordinates first).  With weights over the variables below j, f_0 = 1 - u_j, f_1 = u_j and the carried tensor C Z:
//   q(0) = C / f_0 sum a0 Z0,   q(1) = C / f_1 sum a1 Z1,   Z' = Z0 + (v f_0 / (f_1 (1 - v))) Z1,   C' = C (1 - v) / f_0,
// and q(v) = f_0' q'(0) + f_1' q'(1) of the next round.
//
// What the prover's own comparisons still see: the first round's q(0) and q(1) are sums over the operands, so a claim that is not
// theirs is refused (a lookup's witness is compared with its table before, and A's plain sums are real in every round).  From
// the second carried round on the weighted part of claim = p(0) + p(1) holds by construction: a fold that went wrong on the
// chip is not noticed here but where A(v), B(v) or S(v) are opened against their commitments.  Sums of both halves of both
// tensors would show it (each fold is linear in them), at 1.28 -> 1.46 ms for an element product of 2048 x 11008.
#pragma once
#include <array>
#include <vector>
#include "../../include/grape_hip.h"
#include "fr.hpp"

struct CarriedFactors {
    bool ok = false;                       // every factor has an inverse
    std::vector<Fr> ratio;                 // the table's value of round k (k >= 1; ratio[0] unused)
    std::vector<Fr> at0, at1;              // q(0) and q(1) of round k from its sums (1 for the round in which the weights enter)
    std::vector<Fr> end;                   // S = end[h] * Z for period h of what is left
    std::vector<Fr> inv_v, inv_1v;         // 1 / v_k and 1 / (1 - v_k)

    // u, v: nu coordinates each; rounds: how many carry; low: how many variables' weights are not carried
    CarriedFactors(const Fr* u, const Fr* v, unsigned nu, unsigned rounds, unsigned low) : u_(u), v_(v), nu_(nu) {
        if (rounds == 0 || nu < rounds + low) return;
        const Fr one = Fr::one();
        const unsigned left = nu - rounds;
        // one inversion for all: v_k, 1 - v_k of every round, then u_j, 1 - u_j of the variables low .. nu - 2
        std::vector<Fr> x;
        for (unsigned k = 0; k < rounds; k++) {
            x.push_back(v[nu - 1 - k]);
            x.push_back(one - v[nu - 1 - k]);
        }
        for (unsigned j = low; j + 1 < nu; j++) {
            x.push_back(u[j]);
            x.push_back(one - u[j]);
        }
        std::vector<Fr> before(x.size());
        Fr product = one;
        for (size_t i = 0; i < x.size(); i++) {
            if (x[i].is_zero()) return;
            before[i] = product;
            product = product * x[i];
        }
        std::vector<Fr> inv(x.size());
        Fr rest = product.inverse();
        for (size_t i = x.size(); i-- > 0;) {
            inv[i] = rest * before[i];
            rest = rest * x[i];
        }
        auto inv_u = [&](unsigned j) { return inv[2 * rounds + 2 * (j - low)]; };
        auto inv_1u = [&](unsigned j) { return inv[2 * rounds + 2 * (j - low) + 1]; };
        Fr c = one;
        for (unsigned k = 0; k < rounds; k++) {
            const unsigned j = nu - 1 - k;
            inv_v.push_back(inv[2 * k]);
            inv_1v.push_back(inv[2 * k + 1]);
            if (k == 0) {
                ratio.push_back(Fr::zero());
                at0.push_back(one);
                at1.push_back(one);
                continue;
            }
            ratio.push_back(v[j] * (one - u[j]) * inv_u(j) * inv_1v[k]);
            at0.push_back(c * inv_1u(j));
            at1.push_back(c * inv_u(j));
            c = c * (one - v[j]) * inv_1u(j);
        }
        end.assign(1, c);
        for (unsigned j = low; j < left; j++) {
            const size_t n = end.size();
            end.resize(2 * n);
            for (size_t h = 0; h < n; h++) {
                end[n + h] = end[h] * inv_u(j);
                end[h] = end[h] * inv_1u(j);
            }
        }
        ok = true;
    }
    // q of round k from its values at 0 and 1 and those of the next round's
    std::array<Fr, 3> polynomial(unsigned k, const Fr& q0, const Fr& q1, const Fr& next0, const Fr& next1) const {
        const Fr &un = u_[nu_ - 2 - k], &v = v_[nu_ - 1 - k];
        const Fr at_v = next0 + un * (next1 - next0);
        const Fr top = (q0 + (q1 - q0) * v - at_v) * inv_v[k] * inv_1v[k];
        return {q0, q1 - q0 - top, top};
    }

    // The rounds run two to a pass, an odd one's last alone.
    static uint32_t place_in_pass(unsigned i, unsigned rounds) {
        return i % 2 ? GRAPE_CARRIED_SECOND : i + 1 < rounds ? GRAPE_CARRIED_FIRST : GRAPE_CARRIED_SINGLE;
    }
    static void queue_passes(const grape_carried_args* a, unsigned rounds, grape_stream_t st) {
        for (unsigned i = 0; i < rounds; i++) {
            if (a[i].pair == GRAPE_CARRIED_SINGLE) grape_host::check(grape_carried_queue(&a[i], st), "grape_carried_queue");
            if (a[i].pair == GRAPE_CARRIED_FIRST) grape_host::check(grape_carried_queue_pair(&a[i], &a[i + 1], st), "grape_carried_queue_pair");
        }
    }

private:
    const Fr *u_, *v_;
    unsigned nu_;
};
