// One shot at a time over a shared-state plan (svm_tree_plan.h), as plain
// scalar code: the tables' documented meaning (svm_tree_args.h) applied
// literally, for the CPU test of the planner.
#include <cmath>
#include <complex>
#include <cstdint>
#include <cstring>
#include <vector>

#include "clifft_svm.h"
#include "svm_tree_plan.h"

using namespace csvm;
typedef std::complex<double> cd;

namespace {

struct Rng {
    uint64_t s[4];
    static uint64_t rotl(uint64_t x, int k) { return (x << k) | (x >> (64 - k)); }
    uint64_t next() {
        const uint64_t r = rotl(s[0] + s[3], 23) + s[0], t = s[1] << 17;
        s[2] ^= s[0], s[3] ^= s[1], s[1] ^= s[2], s[0] ^= s[3], s[2] ^= t, s[3] = rotl(s[3], 45);
        return r;
    }
    double uniform() { return (double)(next() >> 11) * 0x1.0p-53; }
};

uint32_t par(uint64_t x) { return (uint32_t)__builtin_popcountll(x) & 1u; }

struct Shot {
    const clifft_program_view* v;
    const TreePlan& P;
    std::vector<cd> st{cd(1, 0)};
    uint32_t choice = 0;
    std::vector<uint32_t> R;  // the response
    Rng rng;
    uint32_t next_noise = 0;
    double p[2] = {0, 0}, num = 0, den = 0;
    size_t next_pass = 0;
    double* ev;
    bool discarded = false;

    uint32_t bits(uint32_t at, uint32_t n) const { return (R[at / 32] >> (at % 32)) & ((1u << n) - 1u); }
    // the row of `units` units from unit r on
    void add_row(uint32_t r, uint32_t units) {
        for (uint32_t e = 4 * r; e < 4 * (r + units); ++e) R.at(P.rows[2 * e] >> 6) ^= P.rows[2 * e + 1];
    }
    void draw(double cur) {
        if (next_noise >= v->num_sites) {
            next_noise = ~0u;
            return;
        }
        const double t = cur - std::log(1.0 - rng.uniform());
        next_noise = 0;
        while (next_noise < v->num_sites && v->hazards[next_noise] <= t) ++next_noise;
    }
    cd entry(const TreePass& q, uint32_t y) const {
        uint32_t s = 0, g = 0;  // s: a byte offset
        for (uint32_t b = 0; b < q.r; ++b)
            if ((y >> b) & 1u) s ^= q.cols[b], g ^= q.colg[b];
        s /= 16;
        cd a = st[s & ((1u << q.r0) - 1u)];
        if (!q.ez_choices) a *= cd(q.ez_tab[s >> q.r0][0], q.ez_tab[s >> q.r0][1]);
        for (uint32_t b = 0; b < q.m && q.ez_choices; ++b)
            if ((s >> (q.r0 + b)) & 1u) {
                const bool c = q.ez_choice[b] >= 0 && ((choice >> q.ez_choice[b]) & 1u);
                a *= cd(q.ez[b][0], c ? -q.ez[b][1] : q.ez[b][1]);
            }
        for (uint32_t j = 0; j < q.ngen; ++j)
            if ((g >> j) & 1u) {
                const TreePhase& ph = P.phases[q.gen_off + j];
                const bool c = ph.choice >= 0 && ((choice >> ph.choice) & 1u);
                a *= cd(ph.pr, c ? -ph.pi : ph.pi);
            }
        // the turn relative to the pair's (quad's) first entry
        const uint32_t free = q.type == TREE_U4 ? q.r - 2 : q.r - 1, corner = y >> free;
        if (corner) {
            const uint32_t bit = 32 - corner;
            uint32_t sg = q.sign0 >> bit;
            for (uint32_t b = 0; b < free; ++b)
                if ((y >> b) & 1u) sg ^= q.cols_s[b] >> bit;
            if (sg & 1u) a = -a;
            if ((q.quarter >> bit) & 1u) a *= cd(0, 1);
        }
        return a;
    }
    void pass(const TreePass& q) {
        const uint32_t half = 1u << (q.r - 1), free = q.type == TREE_U4 ? q.r - 2 : q.r - 1;
        std::vector<cd> w(2 * half);
        const bool ev = q.type == TREE_EV || q.type == TREE_EV0;
        std::vector<uint32_t> seen(2 * half, 0);
        for (uint32_t y = 0; y < 2 * half; ++y) {
            uint32_t o = y >> free << free;  // EXP_VAL sums stay in coordinate order
            for (uint32_t b = 0; b < free; ++b)
                if ((y >> b) & 1u) o ^= q.colo[b] / 16;
            if (ev) o = y;
            seen[o]++;
            w[o] = entry(q, y);
        }
        for (uint32_t n : seen)
            if (n != 1) w[0] = cd(1e300, 0);  // colo is not a permutation
        const double s2 = 0.70710678118654752440;
        p[0] = p[1] = num = den = 0;
        if (q.type == TREE_EV || q.type == TREE_EV0) {
            for (uint32_t i = 0; i < half; ++i) {
                const cd a = w[i], b = w[i + half];
                const double zl = par(i & q.evz) ? -1 : 1, zh = par((i | half) & q.evz) ? -1 : 1;
                den += std::norm(a) + std::norm(b);
                if (q.type == TREE_EV0)
                    num += zl * std::norm(a) + zh * std::norm(b);
                else {
                    const cd l = std::conj(b) * a * zl, h = std::conj(a) * b * zh;
                    num += q.ev_imag ? -(l + h).imag() : (l + h).real();
                }
            }
            num *= q.ev_sign;
            return;
        }
        if (q.type == TREE_U4) {
            const uint32_t n = half / 2;
            const clifft_u4_entry& e = v->u4_nodes[q.node].entries[(choice >> q.choice) & 15u];
            for (uint32_t i = 0; i < n; ++i) {
                cd in[4], o[4];
                for (int c = 0; c < 4; ++c) in[c] = w[i + c * n];
                for (int r = 0; r < 4; ++r)
                    for (int c = 0; c < 4; ++c) o[r] += cd(e.matrix[r][c][0], e.matrix[r][c][1]) * in[c];
                for (int c = 0; c < 4; ++c) w[i + c * n] = o[c];
            }
        }
        for (uint32_t i = 0; i < half; ++i) {
            const cd a = w[i], b = w[i + half];
            if (q.type == TREE_DIAG) {
                p[0] += std::norm(a), p[1] += std::norm(b);
            } else if (q.type == TREE_INTERFERE || q.type == TREE_H) {
                p[0] += std::norm(a + b), p[1] += std::norm(a - b);
                w[i] = (a + b) * s2, w[i + half] = (a - b) * s2;
            } else if (q.type == TREE_U2) {
                const auto& m = v->u2_nodes[q.node].matrices[(choice >> q.choice) & 3u];
                w[i] = cd(m[0][0], m[0][1]) * a + cd(m[1][0], m[1][1]) * b;
                w[i + half] = cd(m[2][0], m[2][1]) * a + cd(m[3][0], m[3][1]) * b;
            }
        }
        st.swap(w);
        if (q.reset) choice = 0;
    }
    void run() {
        R.assign(P.dense.begin(), P.dense.begin() + P.words);
        for (size_t pc = 0; pc + 1 < P.code.size(); ++pc) {
            const clifft_instruction& in = P.code[pc];
            uint64_t w0, w1;
            memcpy(&w0, in.p.raw, 8);
            memcpy(&w1, in.p.raw + 8, 8);
            const uint32_t i0 = (uint32_t)w0, i1 = (uint32_t)(w0 >> 32), n = in.reserved;
            switch (in.opcode) {
                case kLpRandom:
                    for (uint32_t j = 0; j < in.axis_1; ++j)
                        if (!(rng.uniform() < 0.5)) add_row(i1 + j * in.axis_2, in.axis_2);
                    break;
                case kLpNoise:
                    while (next_noise >= i0 && next_noise < i1) {
                        const TreeSite t = P.sites[next_noise];
                        const double u = rng.uniform();
                        for (uint32_t c = t.first; c < t.first + t.n; ++c)
                            if (u * P.chans[t.first + t.n - 1].cum < P.chans[c].cum) {
                                const TreeChan& ch = P.chans[c];
                                if (ch.first & 1) R[0] = 0xDEADBEEF;  // not aligned
                                for (uint32_t e = ch.first; e < ch.first + ch.n; ++e)
                                    R.at(P.chan_rows[2 * e] >> 6) ^= P.chan_rows[2 * e + 1];
                                break;
                            }
                        next_noise++;
                        draw(t.hazard);
                    }
                    break;
                case kLpReadout:
                    for (uint32_t j = 0; j < in.axis_1; ++j)
                        if (rng.uniform() < v->ro_prob[i0 + j]) add_row(i1 + j * in.axis_2, in.axis_2);
                    break;
                case kLpPostselect:
                    if (bits(i0, 1)) {
                        for (uint32_t w = 0; w < P.words; ++w) R[w] &= P.dense[(size_t)i1 * P.words + w];
                        discarded = true;
                        return;
                    }
                    break;
                case kTreeChoice: choice |= bits(i0, n) << w1; break;
                case kTreePass: pass(P.passes[next_pass++]); break;
                case kTreeMeas: {
                    const TreePass& q = P.passes[next_pass++];
                    pass(q);
                    const double tot = p[0] + p[1], eps = 1e-18 * tot;
                    uint32_t o;
                    if (p[1] <= eps) o = 0;
                    else if (p[0] <= eps) o = 1;
                    else o = rng.uniform() * tot < p[0] ? 0 : 1;
                    const uint32_t half = 1u << (q.r - 1);
                    st = std::vector<cd>(st.begin() + (o ? half : 0), st.begin() + (o ? 2 * half : half));
                    if (o) add_row(i1, in.axis_2);
                    break;
                }
                case kTreeNode: {
                    const uint32_t s = bits(i1, n);
                    const uint32_t o = n == 4 ? v->u4_nodes[i0].entries[s].out_state : v->u2_nodes[i0].out_states[s];
                    for (uint32_t b = 0; b < n; ++b)
                        if ((o >> b) & 1) add_row((uint32_t)w1 + b * in.axis_2, in.axis_2);
                    break;
                }
                case kTreeEv: {
                    if (w1 == 0) pass(P.passes[next_pass++]);
                    const double r = w1 == 1 ? 0.0 : w1 == 2 ? 1.0 : (den > 0 ? num / den : 0.0);
                    ev[i0] = std::fmax(-1.0, std::fmin(1.0, bits(i1, 1) ? -r : r));
                    break;
                }
            }
        }
    }
};

}  // namespace

// Samples `shots` shots of the plan; returns the passes planned, or -1 when
// the planner refuses the program.  khist[i]: the rank before instruction i.
extern "C" int tree_sample(const clifft_program_view* v, const int32_t* khist, uint64_t shots, uint64_t seed, uint8_t* meas,
                           uint8_t* det, uint8_t* obs, double* ev) {
    const std::vector<int32_t> kh(khist, khist + v->num_instructions);
    TreePlanner planner(v, kh);
    const TreePlan P = planner.run();
    if (!P.ok) return -1;
    uint64_t zz = seed;
    auto split = [&] {
        uint64_t y = (zz += 0x9e3779b97f4a7c15ULL);
        y = (y ^ (y >> 30)) * 0xbf58476d1ce4e5b9ULL;
        y = (y ^ (y >> 27)) * 0x94d049bb133111ebULL;
        return y ^ (y >> 31);
    };
    for (uint64_t s = 0; s < shots; ++s) {
        Shot S{v, P};
        for (auto& r : S.rng.s) r = split();
        S.ev = ev + s * v->num_exp_vals;
        S.draw(0.0);
        S.run();
        const uint32_t wm = (v->num_measurements + 31) / 32, wd = (v->num_detectors + 31) / 32;
        for (uint32_t i = 0; i < v->num_measurements; ++i) meas[s * v->num_measurements + i] = (uint8_t)S.bits(i, 1);
        for (uint32_t i = 0; i < v->num_detectors; ++i) det[s * v->num_detectors + i] = (uint8_t)S.bits(32 * wm + i, 1);
        for (uint32_t i = 0; i < v->num_observables; ++i)
            obs[s * v->num_observables + i] =
                (uint8_t)(S.bits(32 * (wm + wd) + i, 1) ^ (i < v->num_expected_observables ? v->expected_observables[i] : 0));
    }
    return (int)P.passes.size();
}
