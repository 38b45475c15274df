// svm_tree_plan.h -- host planner of the shared-state executor.
//
// Rewrites a program's bytecode for a team that runs many shots at once and
// keeps one copy of the amplitudes per group of shots ("node") that agree
// on everything the amplitudes depend on (svm_tree.h).  The rank trajectory
// and the array opcodes are static, so all array work is planned here:
//   * permutation and phase opcodes (CNOT, CZ, SWAP, MULTI_*, S, T, ROT) and
//     expansions are never run one at a time.  They are held back as a
//     linear map over GF(2), a phase polynomial and a phase list and become
//     the gather of the next pass: an active measurement, H, U2, U4 or
//     EXP_VAL;
//   * of the Clifford phases a pass applies only what tells the two entries
//     of a pair apart, which is a sign linear in the pair's index and a
//     quarter turn that all pairs share.  What the entries have in common
//     goes on to the next pass: it never interferes, and at the end nothing
//     reads it;
//   * their effect on the Pauli frame becomes frame opcodes, which the
//     caller packs into the lane superinstructions;
//   * where the amplitudes depend on a frame bit that may be set (T, ROT,
//     expansions: p_x; U2, U4: both bits), a kTreeChoice parts the shots.
// Expansions commute with the permutations and phases recorded before them
// (they add the top axis), so a pass always applies expansions first.
// Clifford phases are exact (signs and swaps of parts), so where they are
// applied does not change a rounding.
#pragma once

#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <cmath>
#include <utility>
#include <vector>

#include "clifft_svm.h"
#include "svm_tree_args.h"

namespace csvm {

struct TreePlan {
    bool ok = false;
    std::vector<clifft_instruction> code;  // sampling opcodes; frame opcodes not packed yet
    std::vector<uint8_t> idle;             // frame opcodes that are the identity from the zero frame
    std::vector<TreePass> passes;
    std::vector<TreePhase> phases;
    // per writing pass: bits that may part the shots before it, and its rank
    std::vector<std::pair<uint32_t, uint32_t>> sizes;
};

class TreePlanner {
  public:
    TreePlanner(const clifft_program_view* view, const std::vector<int32_t>& khist) : v(view), kh(khist) {}

    TreePlan run() {
        if (v->words != 1 || v->peak_rank > kTreeMaxRank) return TreePlan();
        for (uint64_t i = 0; i < v->num_instructions; ++i)
            if (!step(v->bytecode[i], (uint32_t)kh[i])) return TreePlan();
        out.ok = true;
        return std::move(out);
    }

  private:
    struct Expand {
        double zr, zi;
        bool phase;
        int choice;
    };
    // An entry turns by i^<w, y> (-1)^Q(y), Q(y) = <l, y> + the sum of
    // y_a y_b over the pairs of the symmetric matrix m.
    struct Turns {
        uint32_t w = 0, l = 0;
        uint32_t m[32] = {};
        void half(uint32_t u, uint32_t v) {  // (-1)^(<u, y> <v, y>)
            l ^= u & v;
            for (uint32_t r = u; r; r &= r - 1) m[__builtin_ctz(r)] ^= v & ~(r & (0u - r));
            for (uint32_t r = v; r; r &= r - 1) m[__builtin_ctz(r)] ^= u & ~(r & (0u - r));
        }
        void quarter(uint32_t u, int q) {  // i^(q <u, y>)
            if (q & 2) l ^= u;
            if (q & 1) {  // i^a i^b = i^(a xor b) (-1)^(ab)
                half(w, u);
                w ^= u;
            }
        }
        // the bilinear form of Q
        uint32_t form(uint32_t x, uint32_t y) const {
            uint32_t f = 0;
            for (uint32_t r = x; r; r &= r - 1) f ^= par(m[__builtin_ctz(r)] & y);
            return f;
        }
        uint32_t value(uint32_t x) const {  // Q(x)
            uint32_t q = par(l & x);
            for (uint32_t r = x; r; r &= r - 1) {
                const uint32_t a = r & (0u - r);
                q ^= par(m[__builtin_ctz(r)] & x & ~(a | (a - 1u)));
            }
            return q;
        }
        // on coordinates of which bit b stands for the old index place[b]
        Turns on(const std::vector<uint32_t>& place) const {
            Turns n;
            for (size_t b = 0; b < place.size(); ++b) {
                n.w |= par(w & place[b]) << b;
                n.l |= value(place[b]) << b;
                for (size_t c = 0; c < place.size(); ++c)
                    if (c != b) n.m[b] |= form(place[b], place[c]) << c;
            }
            return n;
        }
        Turns below(uint32_t bits) const {  // what depends on the low bits alone
            const uint32_t k = (1u << bits) - 1u;
            Turns n;
            n.w = w & k;
            n.l = l & k;
            for (uint32_t b = 0; b < bits; ++b) n.m[b] = m[b] & k;
            return n;
        }
    };
    struct Gen {  // a general phase where <u, y> is odd
        uint32_t u;
        TreePhase ph;
    };

    const clifft_program_view* v;
    const std::vector<int32_t>& kh;
    TreePlan out;
    // The state at logical index y is turns(y) gens(y) times the entry at
    // source index XOR of src over the bits of y: its low r0 bits name the
    // stored entry, those above the pending expansions.
    uint32_t r0 = 0;             // rank of the stored state
    std::vector<uint32_t> src;
    std::vector<Expand> exps;    // pending expansions, oldest first
    Turns turns;
    std::vector<Gen> gens;       // in order
    uint32_t nchoice = 0;        // choice bits in use
    uint32_t splits = 0;         // bits that may have parted the shots so far
    uint64_t mx = 0, mz = 0;     // frame bits that may be nonzero

    static uint32_t par(uint32_t x) { return (uint32_t)__builtin_popcount(x) & 1u; }
    static uint64_t bit(uint32_t q) { return 1ull << q; }
    bool hx(uint32_t q) const { return (mx >> q) & 1ull; }
    bool hz(uint32_t q) const { return (mz >> q) & 1ull; }
    uint32_t rank() const { return r0 + (uint32_t)exps.size(); }

    // ------------------------------------------------------------ emission
    clifft_instruction& emit(const clifft_instruction& in, bool idle = false) {
        out.code.push_back(in);
        out.idle.push_back(idle ? 1 : 0);
        return out.code.back();
    }
    clifft_instruction blank(uint32_t op, uint32_t a1 = 0, uint32_t a2 = 0) {
        clifft_instruction in;
        memset(&in, 0, sizeof(in));
        in.opcode = (uint8_t)op;
        in.axis_1 = (uint16_t)a1;
        in.axis_2 = (uint16_t)a2;
        return in;
    }
    static void word(clifft_instruction& in, int w, uint64_t x) { memcpy(in.p.raw + 8 * w, &x, 8); }
    // a frame opcode, with the bits it may set (the rules of the frame
    // handlers); marked idle when every bit it reads is known zero
    void frame(uint32_t op, uint32_t a, uint32_t b) {
        bool idle = false;
        const bool xa = hx(a), za = hz(a);
        switch (op) {
            case CLIFFT_OP_FRAME_CNOT:
                idle = !xa && !hz(b);
                if (hz(b)) mz |= bit(a);
                if (xa) mx |= bit(b);
                break;
            case CLIFFT_OP_FRAME_CZ: {
                const bool xb = hx(b);
                idle = !xa && !xb;
                if (xa) mz |= bit(b);
                if (xb) mz |= bit(a);
                break;
            }
            case CLIFFT_OP_FRAME_H:
                idle = !xa && !za;
                if (!idle) mx |= bit(a), mz |= bit(a);
                break;
            case CLIFFT_OP_FRAME_S:
            case CLIFFT_OP_FRAME_S_DAG:
                idle = !xa;
                if (xa) mz |= bit(a);
                break;
            default: {  // FRAME_SWAP
                const bool xb = hx(b), zb = hz(b);
                idle = !xa && !za && !xb && !zb;
                const uint64_t m = ~(bit(a) | bit(b));
                mx = (mx & m) | (xb ? bit(a) : 0) | (xa ? bit(b) : 0);
                mz = (mz & m) | (zb ? bit(a) : 0) | (za ? bit(b) : 0);
                break;
            }
        }
        emit(blank(op, a, b), idle);
    }
    // the shots part by `bits` frame bits; their place in the choice word
    int choice(uint32_t a, uint32_t b, uint32_t bits) {
        if (nchoice + bits > kTreeMaxChoice) materialise();
        const int at = (int)nchoice;
        clifft_instruction c = blank(kTreeChoice, a, b);
        c.reserved = (uint8_t)bits;
        word(c, 0, (uint64_t)at);
        emit(c);
        nchoice += bits;
        splits += bits;
        return at;
    }

    // --------------------------------------------------------------- passes
    // A basis of the pair indices (the pair bit stays on top) whose first six
    // vectors, a wavefront's lanes, touch whole 128-byte lines on both sides:
    // alternately the written state's low bits and the pair indices whose
    // sources differ in the stored state's low bits.
    static std::vector<uint32_t> lane_basis(const uint32_t* cols, uint32_t r) {
        const uint32_t t = r - 1;
        std::vector<std::pair<uint32_t, uint32_t>> rows(r);  // (source, coordinate), reduced to unit sources
        for (uint32_t b = 0; b < r; ++b) rows[b] = {cols[b], 1u << b};
        for (uint32_t j = 0; j < r; ++j) {
            size_t k = j;
            while (k < r && !((rows[k].first >> j) & 1u)) ++k;
            if (k == r) return identity(r);  // not invertible: cannot be
            std::swap(rows[j], rows[k]);
            for (uint32_t b = 0; b < r; ++b)
                if (b != j && ((rows[b].first >> j) & 1u)) {
                    rows[b].first ^= rows[j].first;
                    rows[b].second ^= rows[j].second;
                }
        }
        std::vector<uint32_t> out, echelon(t, 0);
        auto add = [&](uint32_t x) {
            uint32_t y = x;
            for (uint32_t b = t; b-- > 0;)
                if (((y >> b) & 1u) && echelon[b]) y ^= echelon[b];
            if (y == 0) return;
            echelon[31 - __builtin_clz(y)] = y;
            out.push_back(x);
        };
        for (uint32_t j = 0; j < t && out.size() < 6; ++j) {
            add(1u << j);
            if (out.size() < 6) add(rows[j].second & ((1u << t) - 1u));
        }
        for (uint32_t j = 0; j < t; ++j) add(1u << j);
        out.push_back(1u << t);
        return out;
    }
    // The pass's signs of corner `bit` (31: the upper entry of a pair), which
    // lies in direction d of the coordinates that t is given on:
    //   turns(y + d) / turns(y) = i^<w, d> (-1)^(Q(d) + B(d, y) + <w, d> <w, y>)
    static void relative(TreePass& p, const Turns& t, uint32_t d, uint32_t free, uint32_t bit, const std::vector<uint32_t>& place) {
        const uint32_t wd = par(t.w & d);
        p.quarter |= wd << bit;
        p.sign0 |= t.value(d) << bit;
        for (uint32_t b = 0; b < free; ++b) p.cols_s[b] |= (t.form(d, place[b]) ^ (wd & par(t.w & place[b]))) << bit;
    }
    // A pass of `type` over coordinates whose bit b is the logical index
    // q[b].  Returns its number; `at`: the turns on these coordinates.
    uint32_t add_pass(uint32_t type, const std::vector<uint32_t>& q, Turns* at = nullptr) {
        TreePass p;
        memset(&p, 0, sizeof(p));
        p.type = type;
        p.r = (uint32_t)q.size();
        put_expansions(p, exps.size());
        for (uint32_t b = 0; b < p.r; ++b)
            for (uint32_t r = q[b]; r; r &= r - 1) p.cols[b] ^= src[__builtin_ctz(r)];
        const std::vector<uint32_t> place = type == TREE_U4 ? identity(p.r) : lane_basis(p.cols, p.r);
        const std::vector<uint32_t> cols(p.cols, p.cols + p.r);
        for (uint32_t b = 0; b < p.r; ++b) {
            p.cols[b] = 0;
            for (uint32_t r = place[b]; r; r &= r - 1) p.cols[b] ^= 16u * cols[__builtin_ctz(r)];
        }
        const Turns t = turns.on(q);
        if (at) *at = t;
        const uint32_t free = type == TREE_U4 ? p.r - 2 : p.r - 1;
        for (uint32_t b = 0; b < free; ++b) p.colo[b] = 16u * place[b];
        if (type == TREE_U4) {
            relative(p, t, 1u << free, free, 31, place);
            relative(p, t, 2u << free, free, 30, place);
            relative(p, t, 3u << free, free, 29, place);
        } else if (type != TREE_COPY && type != TREE_EV0) {
            relative(p, t, 1u << free, free, 31, place);
        }
        p.ngen = (uint32_t)gens.size();
        p.gen_off = (uint32_t)out.phases.size();
        for (size_t j = 0; j < gens.size(); ++j) {
            out.phases.push_back(gens[j].ph);
            for (uint32_t b = 0; b < p.r; ++b) {
                uint32_t y = 0;
                for (uint32_t r = place[b]; r; r &= r - 1) y ^= q[__builtin_ctz(r)];
                p.colg[b] |= par(gens[j].u & y) << j;
            }
        }
        if (type != TREE_EV && type != TREE_EV0) out.sizes.push_back({splits, p.r});
        out.passes.push_back(p);
        return (uint32_t)out.passes.size() - 1;
    }
    // a pass that reads through the oldest n pending expansions
    void put_expansions(TreePass& p, size_t n) {
        p.r0 = r0;
        p.m = (uint32_t)n;
        for (size_t b = 0; b < n; ++b) {
            p.ez[b][0] = exps[b].zr;
            p.ez[b][1] = exps[b].zi;
            p.ez_choice[b] = exps[b].choice;
            if (exps[b].choice >= 0) p.ez_choices = 1;
        }
        for (uint32_t e = 0; e < (1u << n); ++e) {
            double re = 1.0, im = 0.0;
            for (size_t b = 0; b < n; ++b)
                if (((e >> b) & 1u) && exps[b].phase) {
                    const double x = re * exps[b].zr - im * exps[b].zi;
                    im = re * exps[b].zi + im * exps[b].zr;
                    re = x;
                }
            p.ez_tab[e][0] = re;
            p.ez_tab[e][1] = im;
        }
    }
    static std::vector<uint32_t> identity(uint32_t r) {
        std::vector<uint32_t> q(r);
        for (uint32_t b = 0; b < r; ++b) q[b] = 1u << b;
        return q;
    }
    void emit_pass(uint32_t) { emit(blank(kTreePass)); }
    // Write the oldest expansions, in source order, until a pass can read
    // through the rest.
    void trim_expansions() {
        while (exps.size() > kTreeMaxExpand) {
            const size_t n = std::min<size_t>(kTreeMaxExpand, exps.size() - kTreeMaxExpand);
            TreePass p;
            memset(&p, 0, sizeof(p));
            p.type = TREE_COPY;
            p.r = r0 + (uint32_t)n;
            put_expansions(p, n);
            for (uint32_t b = 0; b < p.r; ++b) {
                p.cols[b] = 16u << b;
                p.colo[b] = b + 1 < p.r ? 16u << b : 0u;
            }
            out.sizes.push_back({splits, p.r});
            out.passes.push_back(p);
            emit_pass(0);
            r0 += (uint32_t)n;
            exps.erase(exps.begin(), exps.begin() + n);
        }
    }
    // The pass wrote the state: logical bit b of `rank_after` is now stored
    // bit stored[b], `rest` the turns it left.
    void consumed(uint32_t pass, const std::vector<uint32_t>& stored, const Turns& rest) {
        out.passes[pass].reset = 1;
        exps.clear();
        gens.clear();
        nchoice = 0;
        r0 = (uint32_t)stored.size();
        src = stored;
        turns = rest;
    }
    // the state written out in logical order, every general phase applied
    void materialise() {
        if (rank() == 0) return;
        bool plain = exps.empty() && gens.empty() && nchoice == 0;
        for (uint32_t b = 0; plain && b < rank(); ++b) plain = src[b] == 1u << b;
        if (plain) return;
        trim_expansions();
        const Turns rest = turns;
        const uint32_t r = rank(), p = add_pass(TREE_COPY, identity(r));
        emit_pass(p);
        consumed(p, identity(r), rest);
    }
    // x ^= px where popc(x & pm) is odd (its own inverse)
    void perm(uint32_t pm, uint32_t px) {
        std::vector<uint32_t> q = identity(rank());
        for (uint32_t& y : q)
            if (par(y & pm)) y ^= px;
        std::vector<uint32_t> s(q.size(), 0);
        for (size_t b = 0; b < q.size(); ++b)
            for (uint32_t r = q[b]; r; r &= r - 1) s[b] ^= src[__builtin_ctz(r)];
        src = s;
        turns = turns.on(q);
        for (Gen& g : gens) {
            uint32_t u = 0;
            for (size_t b = 0; b < q.size(); ++b) u |= par(g.u & q[b]) << b;
            g.u = u;
        }
    }
    // coordinates of a pass on axis a: the pair bit on top, the top axis in
    // a's place
    static std::vector<uint32_t> pair_on(uint32_t r, uint32_t a) {
        std::vector<uint32_t> q = identity(r);
        std::swap(q[a], q[r - 1]);
        return q;
    }
    // H or U2 on axis a
    uint32_t single(uint32_t type, uint32_t a) {
        trim_expansions();
        const std::vector<uint32_t> q = pair_on(rank(), a);  // its own inverse
        Turns t;
        const uint32_t p = add_pass(type, q, &t);
        emit_pass(p);
        consumed(p, q, t.below(rank() - 1).on(q));
        return p;
    }

    void meas(const clifft_instruction& in, uint32_t axis, uint32_t pair_axis, bool interfere) {
        trim_expansions();
        const uint32_t r = rank();
        Turns t;
        const uint32_t p = add_pass(interfere ? TREE_INTERFERE : TREE_DIAG, pair_on(r, pair_axis), &t);
        clifft_instruction m = blank(kTreeMeas, axis);
        m.reserved = interfere ? 1 : 0;
        m.flags = in.flags;
        word(m, 0, in.p.classical.classical_idx);
        emit(m);
        consumed(p, identity(r - 1), t.below(r - 1));
        splits += 1;
        mx |= bit(axis);
        mz &= ~bit(axis);
    }
    static bool unit(double re, double im) { return std::fabs(std::hypot(re, im) - 1.0) < 1e-9; }

    bool step(const clifft_instruction& in, uint32_t k) {
        const uint32_t op = in.opcode, a = in.axis_1, b = in.axis_2;
        double zr = 0.70710678118654752440, zi = zr;
        switch (op) {
            case CLIFFT_OP_FRAME_CNOT: case CLIFFT_OP_FRAME_CZ: case CLIFFT_OP_FRAME_SWAP:
                if (a >= 64 || b >= 64) return false;
                frame(op, a, b);
                return true;
            case CLIFFT_OP_FRAME_H: case CLIFFT_OP_FRAME_S: case CLIFFT_OP_FRAME_S_DAG:
                if (a >= 64) return false;
                frame(op, a, 0);
                return true;
            case CLIFFT_OP_ARRAY_CNOT:
                if (a == b) return false;
                perm(1u << a, 1u << b);
                frame(CLIFFT_OP_FRAME_CNOT, a, b);
                return true;
            case CLIFFT_OP_ARRAY_CZ:
                if (a == b) return false;
                turns.half(1u << a, 1u << b);
                frame(CLIFFT_OP_FRAME_CZ, a, b);
                return true;
            case CLIFFT_OP_ARRAY_SWAP:
                if (a == b) return false;
                perm((1u << a) | (1u << b), (1u << a) | (1u << b));
                frame(CLIFFT_OP_FRAME_SWAP, a, b);
                return true;
            case CLIFFT_OP_ARRAY_MULTI_CNOT:
            case CLIFFT_OP_ARRAY_MULTI_CZ: {
                const uint64_t m = in.p.multi_gate.mask & ((1ull << k) - 1ull);
                if ((m >> a) & 1ull) return false;
                if (m == 0) return true;
                if (op == CLIFFT_OP_ARRAY_MULTI_CNOT)
                    perm((uint32_t)m, 1u << a);
                else
                    turns.half(1u << a, (uint32_t)m);
                for (uint64_t r = m; r; r &= r - 1) {
                    const uint32_t c = (uint32_t)__builtin_ctzll(r);
                    if (op == CLIFFT_OP_ARRAY_MULTI_CNOT)
                        frame(CLIFFT_OP_FRAME_CNOT, c, a);
                    else
                        frame(CLIFFT_OP_FRAME_CZ, a, c);
                }
                return true;
            }
            case CLIFFT_OP_ARRAY_S:
            case CLIFFT_OP_ARRAY_S_DAG:
                turns.quarter(1u << a, op == CLIFFT_OP_ARRAY_S ? 1 : 3);
                frame(op == CLIFFT_OP_ARRAY_S ? CLIFFT_OP_FRAME_S : CLIFFT_OP_FRAME_S_DAG, a, 0);
                return true;
            case CLIFFT_OP_ARRAY_T:
            case CLIFFT_OP_ARRAY_T_DAG:
            case CLIFFT_OP_ARRAY_ROT: {
                if (a >= 64) return false;
                if (op == CLIFFT_OP_ARRAY_T_DAG) zi = -zi;
                if (op == CLIFFT_OP_ARRAY_ROT) zr = in.p.math.weight_re, zi = in.p.math.weight_im;
                if (!unit(zr, zi)) return false;
                if (a >= k) return true;  // a phase of gamma
                if (gens.size() == kTreeMaxGen) materialise();
                Gen g;
                memset(&g, 0, sizeof(g));
                g.ph.choice = hx(a) ? choice(a, 0, 1) : -1;
                g.ph.pr = zr;
                g.ph.pi = zi;
                g.u = 1u << a;
                gens.push_back(g);
                return true;
            }
            case CLIFFT_OP_ARRAY_H:
                single(TREE_H, a);
                frame(CLIFFT_OP_FRAME_H, a, 0);
                return true;
            case CLIFFT_OP_ARRAY_U2: {
                if (a >= 64) return false;
                if (a >= k) {
                    // the amplitudes stay; |gamma| must not tell shots apart
                    for (const double* g : {v->u2_nodes[in.p.u.cp_idx].gamma[0], v->u2_nodes[in.p.u.cp_idx].gamma[1],
                                            v->u2_nodes[in.p.u.cp_idx].gamma[2], v->u2_nodes[in.p.u.cp_idx].gamma[3]})
                        if (!unit(g[0], g[1])) return false;
                } else {
                    const int c = choice(a, 0, 2);
                    const uint32_t p = single(TREE_U2, a);
                    out.passes[p].node = in.p.u.cp_idx;
                    out.passes[p].choice = (uint32_t)c;
                }
                clifft_instruction n = blank(kTreeNode, a);
                word(n, 0, in.p.u.cp_idx);
                emit(n);
                mx |= bit(a);
                mz |= bit(a);
                return true;
            }
            case CLIFFT_OP_ARRAY_U4: {
                if (a >= k || b >= k || a == b) return false;
                const int c = choice(a, b, 4);
                trim_expansions();
                const uint32_t r = rank();
                std::vector<uint32_t> q;
                for (uint32_t l = 0; l < r; ++l)
                    if (l != a && l != b) q.push_back(1u << l);
                q.push_back(1u << a);
                q.push_back(1u << b);
                Turns t;
                const uint32_t p = add_pass(TREE_U4, q, &t);
                out.passes[p].node = in.p.u.cp_idx;
                out.passes[p].choice = (uint32_t)c;
                emit_pass(p);
                std::vector<uint32_t> stored(r);
                for (uint32_t l = 0; l < r; ++l) stored[__builtin_ctz(q[l])] = 1u << l;
                consumed(p, stored, t.below(r - 2).on(stored));
                clifft_instruction n = blank(kTreeNode, a, b);
                n.reserved = 1;
                word(n, 0, in.p.u.cp_idx);
                emit(n);
                mx |= bit(a) | bit(b);
                mz |= bit(a) | bit(b);
                return true;
            }
            case CLIFFT_OP_EXPAND:
            case CLIFFT_OP_EXPAND_T:
            case CLIFFT_OP_EXPAND_T_DAG:
            case CLIFFT_OP_EXPAND_ROT: {
                if (a >= 64) return false;
                if (op == CLIFFT_OP_EXPAND_T_DAG) zi = -zi;
                if (op == CLIFFT_OP_EXPAND_ROT) zr = in.p.math.weight_re, zi = in.p.math.weight_im;
                Expand e;
                e.phase = op != CLIFFT_OP_EXPAND;
                if (!e.phase) zr = 1.0, zi = 0.0;
                if (!unit(zr, zi)) return false;
                e.choice = e.phase && hx(a) ? choice(a, 0, 1) : -1;
                e.zr = zr;
                e.zi = zi;
                src.push_back(1u << rank());
                exps.push_back(e);
                return true;
            }
            case CLIFFT_OP_MEAS_ACTIVE_DIAGONAL:
                if (a >= 64) return false;
                meas(in, a, k - 1, false);
                return true;
            case CLIFFT_OP_MEAS_ACTIVE_INTERFERE:
                if (a >= 64) return false;
                meas(in, a, k - 1, true);
                return true;
            case CLIFFT_OP_SWAP_MEAS_INTERFERE:
                if (a >= 64 || b >= 64) return false;
                if (a != b) frame(CLIFFT_OP_FRAME_SWAP, a, b);
                meas(in, b, a == b ? k - 1 : a, true);
                return true;
            case CLIFFT_OP_MEAS_DORMANT_RANDOM:
                if (a >= 64) return false;
                emit(in);
                mx |= bit(a);
                mz &= ~bit(a);
                return true;
            case CLIFFT_OP_MEAS_DORMANT_STATIC:
            case CLIFFT_OP_READOUT_NOISE:
            case CLIFFT_OP_DETECTOR:
            case CLIFFT_OP_POSTSELECT:
            case CLIFFT_OP_OBSERVABLE:
                emit(in);
                return true;
            case CLIFFT_OP_APPLY_PAULI:
                emit(in);
                mx |= v->pauli_x[in.p.pauli.cp_mask_idx];
                mz |= v->pauli_z[in.p.pauli.cp_mask_idx];
                return true;
            case CLIFFT_OP_NOISE:
            case CLIFFT_OP_NOISE_BLOCK: {
                emit(in);
                const uint64_t s0 = in.p.pauli.cp_mask_idx;
                const uint64_t s1 = std::min<uint64_t>(v->num_sites, op == CLIFFT_OP_NOISE ? s0 + 1 : s0 + in.p.pauli.condition_idx);
                for (uint64_t s = s0; s < s1; ++s)
                    for (uint32_t c = v->site_chan_off[s]; c < v->site_chan_off[s + 1]; ++c) {
                        mx |= v->chan_x[c];
                        mz |= v->chan_z[c];
                    }
                return true;
            }
            case CLIFFT_OP_EXP_VAL: {
                const uint32_t ci = in.p.exp_val.cp_exp_val_idx;
                const uint64_t am = (1ull << k) - 1ull, x = v->ev_x[ci], z = v->ev_z[ci];
                uint32_t kind = 0;
                if (x & ~am) {
                    kind = 1;
                } else if (k == 0) {
                    kind = 2;
                } else {
                    const uint32_t xa = (uint32_t)(x & am), za = (uint32_t)(z & am);
                    materialise();
                    std::vector<uint32_t> q = identity(k);
                    if (xa) {
                        const uint32_t p = 31u - (uint32_t)__builtin_clz(xa);
                        q[p] = 1u << (k - 1);
                        q[k - 1] = xa;
                    }
                    const uint32_t pass = add_pass(xa ? TREE_EV : TREE_EV0, q);
                    TreePass& tp = out.passes[pass];
                    for (uint32_t l = 0; l < k; ++l) {
                        uint32_t y = 0;  // the logical index of coordinate bit l
                        for (uint32_t r = l + 1 < k ? tp.colo[l] / 16u : 1u << l; r; r &= r - 1) y ^= q[__builtin_ctz(r)];
                        if (par(y & za)) tp.evz |= 1u << l;
                    }
                    const uint32_t yc = (uint32_t)__builtin_popcount(xa & za) & 3u;
                    tp.ev_imag = yc & 1u;
                    tp.ev_sign = yc >= 2 ? -1 : 1;
                }
                clifft_instruction e = blank(kTreeEv);
                word(e, 0, (uint64_t)ci | ((uint64_t)in.p.exp_val.exp_val_idx << 32));
                word(e, 1, kind);
                emit(e);
                return true;
            }
            default:
                return false;  // *_FORCED in the source, unknown opcodes
        }
    }
};

}  // namespace csvm
