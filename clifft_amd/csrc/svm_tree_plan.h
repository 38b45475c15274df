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
//   * where the amplitudes depend on a frame bit that may be set (T, ROT,
//     expansions: p_x; U2, U4: both bits), a kTreeChoice parts the shots;
//   * the Pauli frame itself, with every opcode that only moves it, becomes
//     the rows by which a shot's random bits flip its response
//     (svm_tree_args.h), found by one backward pass over the program.
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

// The draws x 2^-53 (x: 53 random bits) that are below p are those with x below
// this; none where p is not a number (a quotient of sums that overflowed).
inline uint64_t draw_limit(double p) {
    return p > 0.0 ? (uint64_t)std::ceil(std::min(p, 1.0) * 0x1.0p53) : 0;  // (scaling by 2^53 is exact)
}

struct TreePlan {
    bool ok = false;
    std::vector<clifft_instruction> code, forced;  // the sampled and the forced walk
    std::vector<TreePass> passes;
    std::vector<TreePhase> phases;
    uint32_t words = 0;               // of a shot's response
    std::vector<uint32_t> dense;      // `words` each
    std::vector<uint32_t> rows;       // 8 words a unit
    std::vector<TreeSite> sites;
    std::vector<TreeChan> chans;
    std::vector<uint32_t> chan_rows;  // two words an entry
    bool can_force = false;           // every record slot is visible and written once
    // per writing pass: bits that may part the shots before it, and its rank
    std::vector<std::pair<uint32_t, uint32_t>> sizes;
};

// The response rows: the program (frame opcodes, measurements, noise, and
// the planner's opcodes) taken backward, with the response that an X or a Z
// on each qubit, and each record bit, has from there on.
class ResponsePlanner {
  public:
    ResponsePlanner(const clifft_program_view* view, const std::vector<clifft_instruction>& code, TreePlan& plan)
        : v(view), in(code), out(plan) {}

    bool run() {
        wm = (v->num_measurements + 31) / 32;
        wd = (v->num_detectors + 31) / 32;
        wo = (v->num_observables + 31) / 32;
        if (!single_writers()) return false;
        // bits that are read, each opcode's within one word
        read_at.assign(in.size(), 0);
        uint32_t next = 32 * (wm + wd + wo);
        for (size_t i = 0; i < in.size(); ++i) {
            const uint32_t op = in[i].opcode;
            const uint32_t n = op == kTreeChoice || op == kTreeNode ? in[i].reserved
                               : op == kTreeEv || op == CLIFFT_OP_POSTSELECT ? 1u : 0u;
            if (n == 0) continue;
            if (next % 32 + n > 32) next = (next + 31) / 32 * 32;
            read_at[i] = next;
            next += n;
        }
        W = std::max<uint32_t>((next + 31) / 32, 1);
        if (W > kTreeMaxWords) return false;
        out.words = W;
        const uint32_t nq = 64 * v->words;
        rx.assign(nq, Row(W, 0));
        rz.assign(nq, Row(W, 0));
        rec.assign(v->total_meas_slots, Row(W, 0));
        for (uint32_t i = 0; i < v->num_measurements; ++i) flip(rec[i], i);
        constant.assign(W, 0);
        standing.assign(W, 0);
        for (const clifft_instruction& x : in)
            if (const int64_t bit = writes(x); bit >= 0) standing[bit / 32] |= 1u << (bit % 32);
        out.sites.resize(v->num_sites);
        out.chans.resize(v->num_channels);
        for (uint32_t t = 0; t < v->num_sites; ++t) {
            const uint32_t c0 = v->site_chan_off[t], c1 = v->site_chan_off[t + 1];
            out.sites[t] = {c0, c1 - c0, v->hazards[t]};
            double acc = 0.0;  // in the reference's summation order (svm_kernels.inl:1894-1909)
            for (uint32_t c = c0; c < c1; ++c) out.chans[c] = {acc += v->chan_prob[c], 0, 0};
        }
        std::vector<clifft_instruction> code, forced;
        for (size_t i = in.size(); i-- > 0;) back(i, code, forced);
        std::reverse(code.begin(), code.end());
        std::reverse(forced.begin(), forced.end());
        out.code = merged(code);
        out.forced = forced;
        out.dense = constant;
        for (std::vector<clifft_instruction>* c : {&out.code, &out.forced}) {
            for (clifft_instruction& x : *c) place_rows(x);
            c->push_back(make(kTreePass, 0, 0, 0));  // read ahead, never run
        }
        return true;
    }

  private:
    typedef std::vector<uint32_t> Row;
    const clifft_program_view* v;
    const std::vector<clifft_instruction>& in;
    TreePlan& out;
    uint32_t W = 1, wm = 0, wd = 0, wo = 0;
    std::vector<uint32_t> read_at;
    std::vector<Row> rx, rz, rec;
    Row constant;
    Row standing;  // the bits written before the instruction at hand
    std::vector<Row> all;  // rows by number, until they are laid down

    static void add(Row& a, const Row& b) {
        for (size_t w = 0; w < a.size(); ++w) a[w] ^= b[w];
    }
    static void flip(Row& a, uint32_t bit) { a[bit / 32] ^= 1u << (bit % 32); }
    static void word(clifft_instruction& x, int w, uint64_t y) { memcpy(x.p.raw + 8 * w, &y, 8); }
    uint32_t det_bit(uint32_t i) const { return 32 * wm + i; }
    uint32_t obs_bit(uint32_t i) const { return 32 * (wm + wd) + i; }
    uint32_t add_row(const Row& a) {
        all.push_back(a);
        return (uint32_t)all.size() - 1;
    }
    // Lay down the rows that an instruction names.
    void place_rows(clifft_instruction& x) {
        uint64_t w2;
        memcpy(&w2, x.p.raw + 8, 8);
        uint32_t first = x.p.classical.expected_val, n = 1;
        if (x.opcode == kLpPostselect) {
            x.p.classical.expected_val = (uint32_t)(out.dense.size() / W);
            out.dense.insert(out.dense.end(), all[first].begin(), all[first].end());
            return;
        }
        if (x.opcode == kTreeNode) {
            first = (uint32_t)w2;
            n = x.reserved;
        } else if (x.opcode == kLpRandom || x.opcode == kLpReadout) {
            n = x.axis_1;
        } else if (x.opcode != kLpCoin && x.opcode != kTreeMeas) {
            return;
        }
        size_t most = 1;
        for (uint32_t r = first; r < first + n; ++r) {
            size_t k = 0;
            for (uint32_t m : all[r]) k += m != 0;
            most = std::max(most, k);
        }
        const size_t units = (most + 3) / 4, base = out.rows.size() / 8;
        for (uint32_t r = first; r < first + n; ++r) {
            const size_t end = out.rows.size() + 8 * units;
            entries(all[r], out.rows);
            out.rows.resize(end, 0);
        }
        x.axis_2 = (uint16_t)units;
        if (x.opcode == kTreeNode)
            word(x, 1, base);
        else
            x.p.classical.expected_val = (uint32_t)base;
    }
    static void entries(const Row& a, std::vector<uint32_t>& to) {
        for (uint32_t w = 0; w < a.size(); ++w)
            if (a[w]) {
                to.push_back(w << 6);
                to.push_back(a[w]);
            }
    }
    clifft_instruction make(uint32_t op, uint32_t count, uint64_t i0, uint64_t i1) {
        clifft_instruction x;
        memset(&x, 0, sizeof(x));
        x.opcode = (uint8_t)op;
        x.axis_1 = (uint16_t)count;
        word(x, 0, (i0 & 0xFFFFFFFFu) | (i1 << 32));
        return x;
    }
    // Every record and detector slot has one writer, and no post-selection
    // stands between two terms of an observable: the response then holds each
    // bit's final value, and what a discarded shot leaves is a set of bits.
    // Every noise site has one instruction: its channels keep one row each.
    bool single_writers() {
        std::vector<uint8_t> site(v->num_sites, 0);
        std::vector<uint8_t> m(v->total_meas_slots, 0), d(v->num_detectors, 0), o(v->num_observables, 0);
        bool post = false;
        std::vector<uint8_t> o_post(v->num_observables, 0);
        for (const clifft_instruction& x : in) {
            switch (x.opcode) {
                case CLIFFT_OP_MEAS_DORMANT_STATIC: case CLIFFT_OP_MEAS_DORMANT_RANDOM: case kTreeMeas:
                    if (m[x.p.classical.classical_idx]++) return false;
                    break;
                case CLIFFT_OP_POSTSELECT:
                    for (size_t i = 0; i < o.size(); ++i) o_post[i] = o[i];
                    post = true;
                    if (d[x.p.pauli.condition_idx]++) return false;
                    break;
                case CLIFFT_OP_DETECTOR:
                    if (d[x.p.pauli.condition_idx]++) return false;
                    break;
                case CLIFFT_OP_NOISE:
                case CLIFFT_OP_NOISE_BLOCK: {
                    const uint64_t s0 = x.p.pauli.cp_mask_idx;
                    const uint64_t s1 = std::min<uint64_t>(v->num_sites, x.opcode == CLIFFT_OP_NOISE ? s0 + 1 : s0 + x.p.pauli.condition_idx);
                    for (uint64_t s = s0; s < s1; ++s)
                        if (site[s]++) return false;
                    break;
                }
                case CLIFFT_OP_OBSERVABLE:
                    if (post && o_post[x.p.pauli.condition_idx]) return false;
                    o[x.p.pauli.condition_idx] = 1;
                    break;
            }
        }
        out.can_force = v->total_meas_slots == v->num_measurements;
        for (uint8_t n : m) out.can_force = out.can_force && n == 1;
        return true;
    }
    // the visible bit that an instruction writes, or -1
    int64_t writes(const clifft_instruction& x) const {
        switch (x.opcode) {
            case CLIFFT_OP_MEAS_DORMANT_STATIC: case CLIFFT_OP_MEAS_DORMANT_RANDOM: case kTreeMeas:
                return x.p.classical.classical_idx < v->num_measurements ? x.p.classical.classical_idx : -1;
            case CLIFFT_OP_DETECTOR: return det_bit(x.p.pauli.condition_idx);
            case CLIFFT_OP_OBSERVABLE: return obs_bit(x.p.pauli.condition_idx);
        }
        return -1;
    }
    template <class F>
    void each_bit(const uint64_t* mask, F f) const {
        for (uint32_t w = 0; w < v->words; ++w)
            for (uint64_t r = mask[w]; r; r &= r - 1) f(64 * w + (uint32_t)__builtin_ctzll(r));
    }
    void parity_into(uint32_t list, bool obs, uint32_t bit) {
        const uint32_t* off = obs ? v->obs_off : v->det_off;
        const uint32_t* tgt = obs ? v->obs_tgt : v->det_tgt;
        for (uint32_t j = off[list]; j < off[list + 1]; ++j) flip(rec[tgt[j]], bit);
    }

    void back(size_t i, std::vector<clifft_instruction>& code, std::vector<clifft_instruction>& forced) {
        const clifft_instruction& x = in[i];
        const uint32_t op = x.opcode, a = x.axis_1, b = x.axis_2;
        const uint32_t sign = x.flags & CLIFFT_FLAG_SIGN, idx = x.p.classical.classical_idx;
        auto both = [&](const clifft_instruction& y) {
            code.push_back(y);
            forced.push_back(y);
        };
        if (const int64_t bit = writes(x); bit >= 0) standing[bit / 32] &= ~(1u << (bit % 32));
        switch (op) {
            case CLIFFT_OP_FRAME_CNOT:  // x_b ^= x_a, z_a ^= z_b
                add(rx[a], rx[b]);
                add(rz[b], rz[a]);
                break;
            case CLIFFT_OP_FRAME_CZ:  // z_b ^= x_a, z_a ^= x_b
                add(rx[a], rz[b]);
                add(rx[b], rz[a]);
                break;
            case CLIFFT_OP_FRAME_H:
                rx[a].swap(rz[a]);
                break;
            case CLIFFT_OP_FRAME_S:
            case CLIFFT_OP_FRAME_S_DAG:  // z_a ^= x_a
                add(rx[a], rz[a]);
                break;
            case CLIFFT_OP_FRAME_SWAP:
                if (a != b) {
                    rx[a].swap(rx[b]);
                    rz[a].swap(rz[b]);
                }
                break;
            case CLIFFT_OP_MEAS_DORMANT_STATIC:  // record = x_a ^ sign
                if (!(x.flags & CLIFFT_FLAG_IDENTITY)) add(rx[a], rec[idx]);
                if (sign) add(constant, rec[idx]);
                rec[idx].assign(W, 0);
                forced.push_back(make(kLpStatic, 0, idx, 0));
                break;
            case CLIFFT_OP_MEAS_DORMANT_RANDOM: {  // x_a = m, z_a = 0, record = m ^ sign
                Row m = rx[a];
                add(m, rec[idx]);
                if (sign) add(constant, rec[idx]);
                const uint32_t r = add_row(m);
                code.push_back(make(kLpRandom, 1, 0, r));
                forced.push_back(make(kLpCoin, 1, idx, r));
                rx[a].assign(W, 0);
                rz[a].assign(W, 0);
                rec[idx].assign(W, 0);
                break;
            }
            case kTreeMeas: {  // x_a = m = outcome ^ (x_a or z_a), z_a = 0, record = m ^ sign
                Row m = rx[a];
                add(m, rec[idx]);
                if (sign) add(constant, rec[idx]);
                clifft_instruction y = make(kTreeMeas, 0, idx, add_row(m));
                code.push_back(y);
                y.reserved = 1;
                forced.push_back(y);
                (x.reserved & 1 ? rz : rx)[a] = m;
                (x.reserved & 1 ? rx : rz)[a].assign(W, 0);
                rec[idx].assign(W, 0);
                break;
            }
            case kTreeChoice: {
                clifft_instruction y = make(kTreeChoice, 0, read_at[i], 0);
                y.reserved = x.reserved;
                word(y, 1, x.p.classical.classical_idx);  // place in the choice word
                read_frame(x, read_at[i]);
                both(y);
                break;
            }
            case kTreeNode: {  // the axes' bits become those of the state the node leaves
                clifft_instruction y = make(kTreeNode, 0, idx, read_at[i]);
                y.reserved = x.reserved;
                const uint32_t r = add_row(rx[a]);
                add_row(rz[a]);
                if (x.reserved == 4) {
                    add_row(rx[b]);
                    add_row(rz[b]);
                }
                word(y, 1, r);
                for (uint32_t q : {a, x.reserved == 4 ? b : a}) {
                    rx[q].assign(W, 0);
                    rz[q].assign(W, 0);
                }
                read_frame(x, read_at[i]);
                both(y);
                break;
            }
            case kTreePass:
                both(x);
                break;
            case kTreeEv: {
                const uint32_t ci = x.p.exp_val.cp_exp_val_idx;
                clifft_instruction y = make(kTreeEv, 0, x.p.exp_val.exp_val_idx, read_at[i]);
                memcpy(y.p.raw + 8, x.p.raw + 8, 8);  // kind
                each_bit(v->ev_x + (size_t)ci * v->words, [&](uint32_t q) { flip(rz[q], read_at[i]); });
                each_bit(v->ev_z + (size_t)ci * v->words, [&](uint32_t q) { flip(rx[q], read_at[i]); });
                if (v->ev_sign[ci]) flip(constant, read_at[i]);
                both(y);
                break;
            }
            case CLIFFT_OP_APPLY_PAULI: {
                const size_t m = (size_t)x.p.pauli.cp_mask_idx * v->words;
                Row& r = rec[x.p.pauli.condition_idx];
                each_bit(v->pauli_x + m, [&](uint32_t q) { add(r, rx[q]); });
                each_bit(v->pauli_z + m, [&](uint32_t q) { add(r, rz[q]); });
                break;
            }
            case CLIFFT_OP_NOISE:
            case CLIFFT_OP_NOISE_BLOCK: {
                const uint64_t s0 = x.p.pauli.cp_mask_idx;
                const uint64_t s1 = std::min<uint64_t>(v->num_sites, op == CLIFFT_OP_NOISE ? s0 + 1 : s0 + x.p.pauli.condition_idx);
                if (s0 >= s1) break;
                for (uint32_t c = v->site_chan_off[s0]; c < v->site_chan_off[s1]; ++c) {
                    Row r(W, 0);
                    each_bit(v->chan_x + (size_t)c * v->words, [&](uint32_t q) { add(r, rx[q]); });
                    each_bit(v->chan_z + (size_t)c * v->words, [&](uint32_t q) { add(r, rz[q]); });
                    out.chans[c].first = (uint32_t)(out.chan_rows.size() / 2);
                    entries(r, out.chan_rows);
                    out.chans[c].n = (uint32_t)(out.chan_rows.size() / 2) - out.chans[c].first;
                    if (out.chans[c].n & 1) out.chan_rows.resize(out.chan_rows.size() + 2, 0);
                }
                both(make(kLpNoise, 0, s0, s1));
                break;
            }
            case CLIFFT_OP_READOUT_NOISE:
                both(make(kLpReadout, 1, idx, add_row(rec[v->ro_meas_idx[idx]])));
                break;
            case CLIFFT_OP_DETECTOR:
                parity_into(idx, false, det_bit(x.p.pauli.condition_idx));
                if (x.flags & CLIFFT_FLAG_EXPECTED_ONE) flip(constant, det_bit(x.p.pauli.condition_idx));
                break;
            case CLIFFT_OP_POSTSELECT:
                parity_into(idx, false, read_at[i]);
                if (x.flags & CLIFFT_FLAG_EXPECTED_ONE) flip(constant, read_at[i]);
                both(make(kLpPostselect, 0, read_at[i], add_row(standing)));
                break;
            case CLIFFT_OP_OBSERVABLE:
                parity_into(idx, true, obs_bit(x.p.pauli.condition_idx));
                break;
        }
    }
    // the frame bits of a choice or node, from bit `at` on: p_x (and p_z) of
    // axis_1, then of axis_2
    void read_frame(const clifft_instruction& x, uint32_t at) {
        flip(rx[x.axis_1], at);
        if (x.reserved >= 2) flip(rz[x.axis_1], at + 1);
        if (x.reserved == 4) {
            flip(rx[x.axis_2], at + 2);
            flip(rz[x.axis_2], at + 3);
        }
    }
    // Runs of coin flips and of readout entries become one instruction (their
    // rows lie in program order only if reversed, so they are copied), and so
    // do noise sites that follow one another.
    std::vector<clifft_instruction> merged(const std::vector<clifft_instruction>& code) {
        std::vector<clifft_instruction> o;
        for (size_t i = 0; i < code.size();) {
            const uint32_t op = code[i].opcode;
            auto i0 = [&](size_t j) { return code[j].p.classical.classical_idx; };
            auto i1 = [&](size_t j) { return code[j].p.classical.expected_val; };
            size_t j = i + 1;
            if (op == kLpNoise) {
                while (j < code.size() && code[j].opcode == op && i0(j) == i1(j - 1)) ++j;
                o.push_back(make(kLpNoise, 0, i0(i), i1(j - 1)));
            } else if (op == kLpRandom || op == kLpReadout) {
                while (j < code.size() && j - i < 0xFFFF && code[j].opcode == op && (op == kLpRandom || i0(j) == i0(j - 1) + 1)) ++j;
                uint32_t first = 0;
                for (size_t k = i; k < j; ++k) {
                    const uint32_t at = add_row(Row(all[i1(k)]));
                    if (k == i) first = at;
                }
                o.push_back(make(op, (uint32_t)(j - i), i0(i), first));
            } else {
                o.push_back(code[i]);
            }
            i = j;
        }
        return o;
    }
};

class TreePlanner {
  public:
    TreePlanner(const clifft_program_view* view, const std::vector<int32_t>& khist) : v(view), kh(khist) {}

    TreePlan run() {
        if (v->peak_rank > kTreeMaxRank) return TreePlan();
        mx.assign(v->words, 0);
        mz.assign(v->words, 0);
        for (uint64_t i = 0; i < v->num_instructions; ++i)
            if (!step(v->bytecode[i], (uint32_t)kh[i])) return TreePlan();
        out.ok = ResponsePlanner(v, code, out).run();
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
    std::vector<uint64_t> mx, mz;  // frame bits that may be nonzero
    std::vector<clifft_instruction> code;  // frame opcodes and the planner's

    static uint32_t par(uint32_t x) { return (uint32_t)__builtin_popcount(x) & 1u; }
    static bool has(const std::vector<uint64_t>& m, uint32_t q) { return (m[q / 64] >> (q % 64)) & 1ull; }
    static void set(std::vector<uint64_t>& m, uint32_t q, bool b) {
        m[q / 64] = (m[q / 64] & ~(1ull << (q % 64))) | ((uint64_t)b << (q % 64));
    }
    bool hx(uint32_t q) const { return has(mx, q); }
    bool hz(uint32_t q) const { return has(mz, q); }
    bool on_frame(uint32_t q) const { return q < 64 * v->words; }
    uint32_t rank() const { return r0 + (uint32_t)exps.size(); }

    // ------------------------------------------------------------ emission
    void emit(const clifft_instruction& in) { code.push_back(in); }
    clifft_instruction blank(uint32_t op, uint32_t a1 = 0, uint32_t a2 = 0) {
        clifft_instruction in;
        memset(&in, 0, sizeof(in));
        in.opcode = (uint8_t)op;
        in.axis_1 = (uint16_t)a1;
        in.axis_2 = (uint16_t)a2;
        return in;
    }
    static void word(clifft_instruction& in, int w, uint64_t x) { memcpy(in.p.raw + 8 * w, &x, 8); }
    // a frame opcode, and the bits it may set (the rules of the frame handlers)
    void frame(uint32_t op, uint32_t a, uint32_t b) {
        const bool xa = hx(a), za = hz(a);
        switch (op) {
            case CLIFFT_OP_FRAME_CNOT:
                if (hz(b)) set(mz, a, true);
                if (xa) set(mx, b, true);
                break;
            case CLIFFT_OP_FRAME_CZ: {
                const bool xb = hx(b);
                if (xa) set(mz, b, true);
                if (xb) set(mz, a, true);
                break;
            }
            case CLIFFT_OP_FRAME_H:
                set(mx, a, za);
                set(mz, a, xa);
                break;
            case CLIFFT_OP_FRAME_S:
            case CLIFFT_OP_FRAME_S_DAG:
                if (xa) set(mz, a, true);
                break;
            default: {  // FRAME_SWAP
                const bool xb = hx(b), zb = hz(b);
                set(mx, a, xb);
                set(mx, b, xa);
                set(mz, a, zb);
                set(mz, b, za);
                break;
            }
        }
        emit(blank(op, a, b));
    }
    void any(std::vector<uint64_t>& m, const uint64_t* bits) {
        for (uint32_t w = 0; w < v->words; ++w) m[w] |= bits[w];
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
    void emit_pass() { emit(blank(kTreePass)); }
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
            emit_pass();
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
        emit_pass();
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
        emit_pass();
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
        set(mx, axis, true);
        set(mz, axis, false);
    }
    static bool unit(double re, double im) { return std::fabs(std::hypot(re, im) - 1.0) < 1e-9; }

    bool step(const clifft_instruction& in, uint32_t k) {
        const uint32_t op = in.opcode, a = in.axis_1, b = in.axis_2;
        double zr = 0.70710678118654752440, zi = zr;
        switch (op) {
            case CLIFFT_OP_FRAME_CNOT: case CLIFFT_OP_FRAME_CZ: case CLIFFT_OP_FRAME_SWAP:
                if (!on_frame(a) || !on_frame(b)) return false;
                frame(op, a, b);
                return true;
            case CLIFFT_OP_FRAME_H: case CLIFFT_OP_FRAME_S: case CLIFFT_OP_FRAME_S_DAG:
                if (!on_frame(a)) return false;
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
                if (!on_frame(a)) return false;
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
                if (!on_frame(a)) return false;
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
                n.reserved = 2;
                word(n, 0, in.p.u.cp_idx);
                emit(n);
                set(mx, a, true);
                set(mz, a, true);
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
                emit_pass();
                std::vector<uint32_t> stored(r);
                for (uint32_t l = 0; l < r; ++l) stored[__builtin_ctz(q[l])] = 1u << l;
                consumed(p, stored, t.below(r - 2).on(stored));
                clifft_instruction n = blank(kTreeNode, a, b);
                n.reserved = 4;
                word(n, 0, in.p.u.cp_idx);
                emit(n);
                for (uint32_t q : {a, b}) {
                    set(mx, q, true);
                    set(mz, q, true);
                }
                return true;
            }
            case CLIFFT_OP_EXPAND:
            case CLIFFT_OP_EXPAND_T:
            case CLIFFT_OP_EXPAND_T_DAG:
            case CLIFFT_OP_EXPAND_ROT: {
                if (!on_frame(a)) return false;
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
                if (!on_frame(a)) return false;
                meas(in, a, k - 1, false);
                return true;
            case CLIFFT_OP_MEAS_ACTIVE_INTERFERE:
                if (!on_frame(a)) return false;
                meas(in, a, k - 1, true);
                return true;
            case CLIFFT_OP_SWAP_MEAS_INTERFERE:
                if (!on_frame(a) || !on_frame(b)) return false;
                if (a != b) frame(CLIFFT_OP_FRAME_SWAP, a, b);
                meas(in, b, a == b ? k - 1 : a, true);
                return true;
            case CLIFFT_OP_MEAS_DORMANT_RANDOM:
                if (!on_frame(a)) return false;
                emit(in);
                set(mx, a, true);
                set(mz, a, false);
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
                any(mx, v->pauli_x + (size_t)in.p.pauli.cp_mask_idx * v->words);
                any(mz, v->pauli_z + (size_t)in.p.pauli.cp_mask_idx * v->words);
                return true;
            case CLIFFT_OP_NOISE:
            case CLIFFT_OP_NOISE_BLOCK: {
                emit(in);
                const uint64_t s0 = in.p.pauli.cp_mask_idx;
                const uint64_t s1 = std::min<uint64_t>(v->num_sites, op == CLIFFT_OP_NOISE ? s0 + 1 : s0 + in.p.pauli.condition_idx);
                for (uint64_t s = s0; s < s1; ++s)
                    for (uint32_t c = v->site_chan_off[s]; c < v->site_chan_off[s + 1]; ++c) {
                        any(mx, v->chan_x + (size_t)c * v->words);
                        any(mz, v->chan_z + (size_t)c * v->words);
                    }
                return true;
            }
            case CLIFFT_OP_EXP_VAL: {
                const uint32_t ci = in.p.exp_val.cp_exp_val_idx;
                const uint64_t am = (1ull << k) - 1ull;
                const uint64_t x = v->ev_x[(size_t)ci * v->words], z = v->ev_z[(size_t)ci * v->words];
                bool dormant = (x & ~am) != 0;
                for (uint32_t w = 1; w < v->words; ++w) dormant = dormant || v->ev_x[(size_t)ci * v->words + w];
                uint32_t kind = 0;
                if (dormant) {
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
