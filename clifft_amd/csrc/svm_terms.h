// svm_terms.h -- expectation values and gradients of a parameterised program
// as sums of products of sines and cosines of its angles.
//
// A probe P after a Clifford operation C is the probe C^-1 P C before it;
// after a phase diag(1, e^{ia}) on an axis it stays as it is if it has I or Z
// there, and X becomes cos a X - sin a Y, Y becomes cos a Y + sin a X; and the
// new axis of an expansion, (1, e^{ia}) / sqrt 2, contributes 1 for I, 0 for
// Z, cos a for X and sin a for Y.  Taken back to the start of the program a
// probe therefore is
//     <P> = sum over terms  coef * prod cos a_i * prod sin a_j
// with coef from the signs and the fixed phases: no state is needed, where the
// adjoint sweeps (svm_adjoint.h) move 2^rank amplitudes some times per
// operation.  Each phase that a probe does not commute with doubles its
// terms, so this form is taken only where the terms are the smaller work.
#pragma once

#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "clifft_svm.h"

namespace csvm {

struct AdjTerm {
    double coef;
    uint64_t cos_of, sin_of;  // parameters, by bit; the angle's sign is psign's
    uint32_t probe;           // output index
    uint32_t pad;
};

// Arguments of the kernel (svm_terms.hip).
struct TermArgs {
    const double* thetas;     // [batch x num_params]
    const double* psign;      // [num_params]
    const double* coeffs;     // [num_ev] (gradients)
    double* ev_out;           // [batch x num_ev] or null
    double* grad_out;         // [batch x num_params] or null
    const AdjTerm* terms;     // ascending by probe
    const uint32_t* first;    // [num_ev + 1]: each probe's terms
    // [num_ev]: parameters whose phase the state holds at the probe, none where
    // the probe is 0 for its X on a dormant axis
    const uint64_t* before;
    uint64_t active;          // parameters that turn some axis of the state
    uint64_t batch;
    uint32_t num_params, num_ev, num_terms, pad;
};

// Terms up to which their sums are taken instead of the state: half of what
// makes the two equal.  Measured on one MI355X at 16 and at 512 angle vectors
// (rank 6 to 14, one X probe over all axes whose terms double with every
// second rotation; random programs of rank 1 to 12): the terms take 6 us and
// 20 ns a term + 5.5 ns a term and parameter (1064 terms of 16 parameters
// 110 us, 4148 of 26 540, 2845 of 4 171), the sweeps of `ops` operations 2 to
// 2.2 us an operation to rank 8, 3.6 and 5.6 at rank 10 and 12 (16 vectors) and
// 9.5 to 39 at rank 14 (16 and 512 vectors).
inline size_t term_limit(size_t ops, uint32_t rank, uint32_t num_params) {
    const double sweeps = (double)ops * (2.0 + std::ldexp(0.4e-3, (int)rank));
    const double even = (sweeps - 6.0) / (20e-3 + 5.5e-3 * num_params);
    return (size_t)std::min(std::max(0.5 * even, 0.0), 65536.0);
}

struct TermPlan {
    bool ok = false;
    std::vector<AdjTerm> terms;
    std::vector<uint32_t> first;
    std::vector<uint64_t> before;
    uint64_t active = 0;
};

class TermPlanner {
  public:
    // rank[i]: the active rank before instruction i; slot_of[i]: its
    // parameter, or -1
    TermPlanner(const clifft_instruction* code, size_t n, const int32_t* rank, const int32_t* slot_of, uint32_t num_params,
                uint32_t num_ev, const uint64_t* ev_x, const uint64_t* ev_z, const uint8_t* ev_sign, uint32_t words)
        : code(code), n(n), rank(rank), slot_of(slot_of), np(num_params), nev(num_ev), ev_x(ev_x), ev_z(ev_z),
          ev_sign(ev_sign), W(words) {}

    // not ok: an operation without this form (U2, U4, a phase that is not of
    // unit modulus), more than 64 parameters, an output written never or
    // twice, more than `limit` terms, or more than kPathsPerTerm times as many
    // paths: a term that becomes 0 on its way has cost as much as one that
    // stays, and a probe of which none stay would else be expanded in full,
    // doubling at every phase it does not commute with
    TermPlan run(size_t limit) {
        TermPlan out;
        paths_left = kPathsPerTerm * limit;
        if (np > 64) return out;
        std::vector<int64_t> at(nev, -1);  // the instruction of each output
        for (size_t i = 0; i < n; ++i) {
            const clifft_instruction& x = code[i];
            switch (x.opcode) {
                case CLIFFT_OP_ARRAY_U2: case CLIFFT_OP_ARRAY_U4: return out;
                case CLIFFT_OP_EXP_VAL: {
                    int64_t& a = at[x.p.exp_val.exp_val_idx];
                    if (a >= 0) return out;
                    a = (int64_t)i;
                    break;
                }
                case CLIFFT_OP_ARRAY_ROT: case CLIFFT_OP_EXPAND_ROT: {
                    if (slot_of[i] >= 0) {
                        if (x.opcode == CLIFFT_OP_EXPAND_ROT || x.axis_1 < rank[i]) out.active |= 1ull << slot_of[i];
                        break;
                    }
                    double zr, zi;
                    payload(x, zr, zi);
                    if (!(std::fabs(zr * zr + zi * zi - 1.0) < 4e-15)) return out;
                    break;
                }
            }
        }
        for (uint32_t j = 0; j < nev; ++j) {
            if (at[j] < 0) return out;
            out.first.push_back((uint32_t)out.terms.size());
            if (!probe((size_t)at[j], j, limit, out)) return out;
        }
        out.first.push_back((uint32_t)out.terms.size());
        out.ok = true;
        return out;
    }

  private:
    struct Pauli {
        size_t pc;  // instructions [0, pc) are still to be taken
        uint64_t x, z;
        AdjTerm t;
    };
    const clifft_instruction* code;
    size_t n;
    const int32_t *rank, *slot_of;
    uint32_t np, nev;
    const uint64_t *ev_x, *ev_z;
    const uint8_t* ev_sign;
    uint32_t W;
    // Compiled circuits of 9 to 24 qubits and up to 33 probes open 0 to 2.6
    // paths a term; refusing at 8 takes 0.4 ms at a limit of 400 terms.
    static constexpr size_t kPathsPerTerm = 8;
    size_t paths_left = 0;  // that may still be opened

    static void payload(const clifft_instruction& x, double& zr, double& zi) {
        memcpy(&zr, x.p.raw, 8);
        memcpy(&zi, x.p.raw + 8, 8);
    }

    bool probe(size_t at, uint32_t j, size_t limit, TermPlan& out) {
        uint64_t held = 0;
        for (size_t i = 0; i < at; ++i)
            if (slot_of[i] >= 0 && ((out.active >> slot_of[i]) & 1u)) held |= 1ull << slot_of[i];
        const uint32_t ci = code[at].p.exp_val.cp_exp_val_idx, k = (uint32_t)rank[at];
        const uint64_t on = k >= 64 ? ~0ull : (1ull << k) - 1ull;
        bool dormant = (ev_x[(size_t)ci * W] & ~on) != 0;
        for (uint32_t w = 1; w < W; ++w) dormant = dormant || ev_x[(size_t)ci * W + w];
        out.before.push_back(dormant ? 0 : held);
        if (dormant) return true;  // X on a dormant axis: no terms
        std::vector<Pauli> todo(1);
        todo[0] = {at, ev_x[(size_t)ci * W] & on, ev_z[(size_t)ci * W] & on, {ev_sign[ci] ? -1.0 : 1.0, 0, 0, j, 0}};
        while (!todo.empty()) {
            Pauli p = todo.back();
            todo.pop_back();
            bool live = true;
            while (live && p.pc > 0) {
                const size_t waiting = todo.size();
                live = back(p, todo);
                const size_t opened = todo.size() - waiting;
                if (opened > paths_left) return false;
                paths_left -= opened;
            }
            if (!live) continue;
            if (out.terms.size() >= limit) return false;
            out.terms.push_back(p.t);
        }
        return true;
    }

    // Take instruction p.pc - 1; a second term goes to `todo`.  false: p is 0.
    bool back(Pauli& p, std::vector<Pauli>& todo) const {
        const size_t i = --p.pc;
        const clifft_instruction& c = code[i];
        const uint32_t op = c.opcode, a = c.axis_1, b = c.axis_2, k = (uint32_t)rank[i];
        auto bit = [](uint64_t m, uint32_t q) { return (m >> q) & 1ull; };
        auto flip = [&](uint64_t odd) {
            if (odd) p.t.coef = -p.t.coef;
        };
        auto cnot = [&](uint32_t from, uint32_t to) {
            flip(bit(p.x, from) & bit(p.z, to) & (bit(p.x, to) ^ bit(p.z, from) ^ 1ull));
            p.x ^= bit(p.x, from) << to;
            p.z ^= bit(p.z, to) << from;
        };
        auto cz = [&](uint32_t u, uint32_t v) {
            flip(bit(p.x, u) & bit(p.x, v) & (bit(p.z, u) ^ bit(p.z, v)));
            p.z ^= bit(p.x, u) << v;
            p.z ^= bit(p.x, v) << u;
        };
        // the phase's cosine and sine, fixed or a parameter's
        const bool fixed = op == CLIFFT_OP_ARRAY_T || op == CLIFFT_OP_ARRAY_T_DAG || op == CLIFFT_OP_EXPAND_T ||
                           op == CLIFFT_OP_EXPAND_T_DAG || op == CLIFFT_OP_EXPAND || slot_of[i] < 0;
        double zr = 1.0, zi = 0.0;
        if (op == CLIFFT_OP_ARRAY_ROT || op == CLIFFT_OP_EXPAND_ROT) {
            if (fixed) payload(c, zr, zi);
        } else if (op != CLIFFT_OP_EXPAND) {
            zr = 0.70710678118654752440;
            zi = op == CLIFFT_OP_ARRAY_T_DAG || op == CLIFFT_OP_EXPAND_T_DAG ? -zr : zr;
        }
        auto times_cos = [&](Pauli& q) {
            if (fixed) q.t.coef *= zr;
            else q.t.cos_of |= 1ull << slot_of[i];
            return q.t.coef != 0.0;
        };
        auto times_sin = [&](Pauli& q) {
            if (fixed) q.t.coef *= zi;
            else q.t.sin_of |= 1ull << slot_of[i];
            return q.t.coef != 0.0;
        };
        switch (op) {
            case CLIFFT_OP_ARRAY_CNOT: cnot(a, b); break;
            case CLIFFT_OP_ARRAY_CZ: cz(a, b); break;
            case CLIFFT_OP_ARRAY_SWAP: {
                const uint64_t dx = bit(p.x, a) ^ bit(p.x, b), dz = bit(p.z, a) ^ bit(p.z, b);
                if (a != b) {
                    p.x ^= (dx << a) | (dx << b);
                    p.z ^= (dz << a) | (dz << b);
                }
                break;
            }
            case CLIFFT_OP_ARRAY_MULTI_CNOT:
            case CLIFFT_OP_ARRAY_MULTI_CZ: {
                uint64_t m;
                memcpy(&m, c.p.raw, 8);
                if (op == CLIFFT_OP_ARRAY_MULTI_CZ && bit(m, a)) flip(bit(p.x, a));  // Z on the axis itself
                for (m &= ((1ull << k) - 1ull) & ~(1ull << a); m; m &= m - 1) {
                    const uint32_t q = (uint32_t)__builtin_ctzll(m);
                    if (op == CLIFFT_OP_ARRAY_MULTI_CNOT) cnot(q, a);
                    else cz(q, a);
                }
                break;
            }
            case CLIFFT_OP_ARRAY_H: {
                flip(bit(p.x, a) & bit(p.z, a));
                const uint64_t d = bit(p.x, a) ^ bit(p.z, a);
                p.x ^= d << a;
                p.z ^= d << a;
                break;
            }
            case CLIFFT_OP_ARRAY_S:  // X to -Y, Y to X
                flip(bit(p.x, a) & (bit(p.z, a) ^ 1ull));
                p.z ^= bit(p.x, a) << a;
                break;
            case CLIFFT_OP_ARRAY_S_DAG:  // X to Y, Y to -X
                flip(bit(p.x, a) & bit(p.z, a));
                p.z ^= bit(p.x, a) << a;
                break;
            case CLIFFT_OP_ARRAY_T:
            case CLIFFT_OP_ARRAY_T_DAG:
            case CLIFFT_OP_ARRAY_ROT: {
                if (a >= k || !bit(p.x, a)) break;
                Pauli q = p;  // the sine's: X to -Y, Y to X
                if (!bit(q.z, a)) q.t.coef = -q.t.coef;
                q.z ^= 1ull << a;
                if (times_sin(q)) todo.push_back(q);
                return times_cos(p);
            }
            case CLIFFT_OP_EXPAND:
            case CLIFFT_OP_EXPAND_T:
            case CLIFFT_OP_EXPAND_T_DAG:
            case CLIFFT_OP_EXPAND_ROT: {  // its axis is the last one, k
                const uint64_t x = bit(p.x, k), z = bit(p.z, k);
                p.x &= ~(1ull << k);
                p.z &= ~(1ull << k);
                if (!x) return !z;
                return z ? times_sin(p) : times_cos(p);
            }
            default: break;  // frame operations act on the zero frame only
        }
        return true;
    }
};

}  // namespace csvm
