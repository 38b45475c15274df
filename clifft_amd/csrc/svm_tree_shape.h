// svm_tree_shape.h -- the shared-state executor's rules of dispatch: whether a
// program's shots are better off there, on teams of how many threads, and with
// how many shots a team.  Host code without HIP.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <utility>
#include <vector>

#include "clifft_svm.h"
#include "svm_tree_args.h"

namespace csvm {

// Amplitude buffers up to this many entries (each of a team's two) stay in LDS.
constexpr uint64_t kTreeLdsElems = 2048;
// Dynamic LDS limit of its kernels (less the queue head and the block-wide
// "or" the runtime's library keeps in static LDS), and a compute unit's LDS.
constexpr size_t kTreeMaxDynLds = 158 * 1024;
constexpr size_t kTreeCuLds = 160 * 1024;

constexpr uint32_t kTreeChunks = 11;  // shots a team: powers of two to 1024

// Entries of each amplitude buffer of a team, and those all its passes visit.
struct TreeWork {
    uint64_t elems = 1, visited = 0;
};

// What the rules know of a program.
struct TreeProfile {
    bool ok = false;            // it has a plan
    uint32_t code = 0;          // the plan's instructions
    uint32_t words = 0;         // of a shot's response
    uint32_t frame_words = 1;   // 64 qubits each
    uint32_t peak_rank = 0;
    uint32_t instructions = 0;  // the program's
    uint32_t operations = 0;    // those that do not only move frames
    uint32_t arrays = 0;        // those on amplitudes
    double noise = 0.0;         // events a shot has on average
    uint32_t passes = 0;        // that write
    TreeWork work[kTreeChunks];

    void set_program(const clifft_program_view* v) {
        frame_words = v->words;
        peak_rank = v->peak_rank;
        instructions = (uint32_t)v->num_instructions;
        noise = v->num_sites ? v->hazards[v->num_sites - 1] : 0.0;
        for (uint64_t i = 0; i < v->num_instructions; ++i) {
            const uint32_t op = v->bytecode[i].opcode;
            operations += op > CLIFFT_OP_FRAME_SWAP;
            arrays += (op >= CLIFFT_OP_ARRAY_CNOT && op <= CLIFFT_OP_EXPAND_ROT) || op == CLIFFT_OP_MEAS_ACTIVE_DIAGONAL ||
                      op == CLIFFT_OP_MEAS_ACTIVE_INTERFERE || op == CLIFFT_OP_SWAP_MEAS_INTERFERE || op == CLIFFT_OP_EXP_VAL;
        }
    }

    // from (bits that may part the shots, rank) of every writing pass: over N
    // nodes of rank r it writes N 2^r, and before it at most min(chunk, 2^bits)
    // groups of shots can have parted
    void set_passes(const std::vector<std::pair<uint32_t, uint32_t>>& sizes) {
        passes = (uint32_t)sizes.size();
        for (uint32_t e = 0; e < kTreeChunks; ++e) {
            work[e] = TreeWork();
            for (const auto& sr : sizes) {
                const uint64_t entries = 1ull << (std::min(e, sr.first) + sr.second);
                work[e].elems = std::max(work[e].elems, entries);
                work[e].visited += entries;
            }
        }
    }
};
inline const TreeWork& tree_work(const TreeProfile& p, uint32_t chunk) { return p.work[__builtin_ctz(chunk)]; }

struct TreeShape {
    uint32_t threads = 0, chunk = 0;  // of a team: threads, shots
    uint32_t elems = 0;               // entries of each of its two buffers
    size_t lds = 0;                   // bytes
    bool global = false;              // the buffers are in memory, not in LDS
};

// The shape of a team of `chunk` shots on `threads` threads, each with room
// for `faults` forced faults; false where its tables do not fit.
inline bool tree_team(const TreeProfile& p, uint32_t threads, uint32_t chunk, uint32_t faults, TreeShape& s) {
    const TreeWork& w = tree_work(p, chunk);
    if (w.elems > (1ull << 31)) return false;
    s.threads = threads;
    s.chunk = chunk;
    s.elems = (uint32_t)w.elems;
    s.lds = tree_lds_bytes(threads, chunk, p.words + 5 * faults);
    s.global = w.elems > kTreeLdsElems;
    if (!s.global) s.lds += 32u * (size_t)w.elems;
    return s.lds <= kTreeMaxDynLds;
}

// Estimated time (us) of one chunk on a team of shape s that shares its CU
// with `teams` - 1 others: the walk, the passes' fixed part, and the entries
// visited at what the wavefronts in flight reach (fitted to a sweep of team
// sizes and chunks at peak 0 to 16 on one MI355X).
inline double tree_team_us(const TreeProfile& p, const TreeShape& s, double teams) {
    const double waves = s.threads / 64.0, per_simd = teams * waves / 4.0;
    const double walk = 5.0 + 0.35 * p.code + (2.0 + 0.3 * std::log2(waves)) * p.passes;
    const double visited = (double)tree_work(p, s.chunk).visited;
    const double entry = (s.global ? 0.32e-3 : 0.25e-3) * std::max(512.0 / s.threads, teams);
    return walk * (1.0 + 0.18 * std::max(0.0, per_simd - 1.0)) + visited * entry;
}
// ... and of `shots` shots on `cus` compute units: the teams' own time or, where
// it is longer, that of the memory, which is the same for many shapes; `tie`
// then decides between those (0: the teams' own is the longer).
struct TreeTime {
    double us = 0.0, tie = 0.0;
};

// The tie: shapes whose teams are the faster by themselves use the memory the
// better, so 5.5 % of the difference is taken off (the last round without its
// idle places, which the memory fills).  Where that is the same too, the memory's
// time counts 0.2 % more for each halving of the threads below 512 and, without
// noise, 0.26 % for each doubling of a team's shots: all frame bits count as
// parting these, but noise parts few of them, so that more shots are fewer nodes,
// while outcomes and coins part them all, and smaller buffers leave no compute
// unit idle.  (All shapes of 222 calls, peak 8 to 21, 100 to 80000 shots, with
// noise, with resets and with neither.  The first shape of the least time, 64
// threads and the most shots where frame bits part them, took 1.35 times the
// best shape's time on average, 2.8 at most, and up to 1.7 times the per-shot
// executors'.  With the tie 1.06 and 2.0, and nowhere above the first shape; at
// 4.5 to 9 %, all three in proportion, by 1 % at most.  If the tie also takes
// shapes whose own time is longer, up to 20 % above it where both times are
// alike.  5 % for the threads and nothing for the shots: 22 % above it where
// 11054 shots with resets were put 64 to a team, so that 83 compute units had
// none.)
inline TreeTime tree_time(const TreeProfile& p, const TreeShape& s, uint64_t shots, double cus) {
    const double teams = std::ceil((double)shots / s.chunk);
    const double per_cu = std::max(1.0, std::floor(std::min((double)kTreeCuLds / (double)s.lds, 1024.0 / s.threads)));
    const double rounds = std::max(1.0, teams / (cus * per_cu));
    const double visited = (double)tree_work(p, s.chunk).visited;
    // all teams together move 32 B an entry beyond the caches
    const double bytes = s.global ? std::min(teams, cus * per_cu) * 32.0 * (double)s.elems : 0.0;
    const double memory = bytes > 64e6 ? teams * visited * 32.0 / 4.0e6 : 0.0;
    const double team = tree_team_us(p, s, std::min(per_cu, std::ceil(teams / cus)));
    const double own = std::ceil(rounds) * team;
    if (own >= memory) return {own, 0.0};
    const double halvings = std::max(0.0, std::log2(512.0 / s.threads)), doublings = std::log2((double)s.chunk);
    const double even = memory * (1.0 + 0.002 * halvings + (p.noise > 0.0 ? 0.0 : 0.0026) * doublings);
    return {memory, even - 0.055 * (even - rounds * team)};
}

// Estimated time (us) of `shots` shots on the per-shot executors at peak 8 to
// 10: one shot's walk, 1 us an operation, until the wavefronts are more than
// the device holds at once (18 programs of 150 to 700 instructions, 1 to 30000
// shots; an operation is any instruction but a frame one).
inline double per_shot_us(const TreeProfile& p, uint64_t shots) {
    const double many = (double)shots * (p.peak_rank > 9 ? 1.6e-3 : 0.8e-3);
    return 20.0 + (double)p.operations * std::max(1.0, many);
}

// Estimated time (us) of `shots` shots one a lane, to peak 6: one walk, or what
// the lanes in flight give (46 random, memory and Clifford+T programs of 100 to
// 3300 instructions, 1 to 300000 shots: 0.6 to 1.4 times the measured time).
inline double lanes_us(const TreeProfile& p, uint64_t shots, double cus) {
    const double frames = (double)p.instructions - p.operations, rest = (double)p.operations - p.arrays;
    const double amps = std::ldexp((double)p.arrays, (int)p.peak_rank);
    const double walk = 24.0 + 0.032 * frames + 0.27 * rest + 0.6 * p.arrays + 0.0125 * amps;
    const double shot = 0.028 + 0.45e-3 * p.operations + 0.2e-3 * amps + 0.03 * p.noise;
    return std::max(1.1 * walk, (double)shots / cus * shot);
}

// Whether `shots` shots of a program are better off sharing their states.
// Measured on one MI355X, per-shot executors against this one (100 to 300000
// shots): surface-code memories 1.3 to 3 times faster to 49 qubits (25 rounds
// of distance 3 with 300000 shots: the same), 14 to 470 times beyond 64;
// 24-qubit Clifford+T at peak 8 to 14 2 to 300 times, with noise that parts the
// shots at their T gates 1.04 to 25 times at peak 8 to 19; random programs, whose
// frames part almost every shot, 1.1 to 14 times from peak 11 on.  Below that a
// program with a pass for every few instructions can lose (random, 300
// instructions, 60 passes: 0.72 to 0.94 times at peak 1 to 7), so it has to
// beat the lanes' walk, 0.48 us an instruction there, with more shots lanes_us,
// and at peak 8 to 10 per_shot_us (tree_shape).
// `mode`: CLIFFT_SHARED_STATE (0 never, 2 wherever there is a plan).
inline bool tree_better(const TreeProfile& p, uint64_t shots, int mode) {
    if (!p.ok || mode == 0) return false;
    if (mode == 2 || p.frame_words > 1 || p.peak_rank >= 8) return true;
    if (p.peak_rank == 7 && shots >= 4096) return true;
    return 5.0 + 0.35 * p.code + 2.0 * p.passes <= 0.48 * (double)p.instructions;
}

// Entries of a team's buffer up to which more shots may be put into it: where
// frame bits part the shots, nodes grow with the shots at every rank, and one
// such program would take tens of GiB of scratch (a batch of 512 took 99 GB
// for the one with 2^24 entries a team); smaller chunks are the faster ones
// there (random programs, peak 12 x 20000 shots: 5.6 ms at 2^18 entries a
// team, 3.1 ms at 2^15).
inline uint64_t tree_room(const TreeProfile& p) { return std::max<uint64_t>(1ull << 18, 1ull << p.peak_rank); }

// The shape for a launch of `shots` shots: the team size and the shots per
// team of the least time or, if that is the memory's, of the least tie.  False:
// the program has no plan, or the per-shot executors are faster.
inline bool tree_shape(const TreeProfile& p, uint64_t shots, uint32_t faults, uint32_t cus, int mode, TreeShape& best) {
    if (!tree_better(p, shots, mode)) return false;
    TreeTime least, tied;
    TreeShape even;
    bool found = false;
    for (uint32_t threads : {64u, 128u, 256u, 512u, 1024u})
        for (uint32_t chunk = threads; chunk >= 1; chunk /= 2) {
            if (chunk > 2 * shots && chunk > 1) continue;
            TreeShape s;
            if (!tree_team(p, threads, chunk, faults, s) || (chunk > 1 && s.elems > tree_room(p))) continue;
            const TreeTime t = tree_time(p, s, shots, cus);
            if (!found || t.us < least.us) best = s, least = t;
            if (t.tie > 0.0 && (tied.tie == 0.0 || t.tie < tied.tie)) even = s, tied = t;
            found = true;
        }
    if (least.tie > 0.0) best = even, least = tied;
    const double cost = least.us;
    if (!found || mode != 1 || faults || p.frame_words > 1) return found;
    // (random, 400 instructions, 95 passes, peak 10: 375 us against 310 at 1 to
    // 100 shots, 400 against 520 at 1000)
    if (p.peak_rank >= 8 && p.peak_rank <= 10) return 1.1 * cost <= per_shot_us(p, shots);
    // The estimate leaves out the noise events and, where every compute unit has
    // several teams, is the lower the smaller these are: by 1.4 at 64 threads,
    // high by 1.25 at 1024, but not in memory (the others' factors here are a
    // tenth less).  (Random, 300 instructions, 300000 shots, peak 1 to 5: 1.3 to
    // 3 times as slow as lanes.)
    if (p.peak_rank <= 6 && shots >= 4096) {
        const double low = best.threads == 64 ? 1.25 : best.threads == 128 ? 1.05 : best.threads == 256 ? 0.95 : best.global ? 1.0 : best.threads == 512 ? 0.8 : 0.7;
        return low * cost + 0.045 * p.noise * (double)shots / cus <= lanes_us(p, shots, cus);
    }
    return true;
}

// Estimated time (us) of a batch's `total` shots one shot a lane, to peak 6, if
// all its programs were like this one: one walk, or what the lanes in flight
// give (fitted to batches of 8 to 256 random programs, 100 to 8000 shots each,
// at peak 3 to 6: 0.7 to 1.2 times the measured time).
inline double batch_lanes_us(const TreeProfile& p, uint64_t total, double cus) {
    const double frames = (double)p.instructions - p.operations, amps = std::ldexp(1.0, (int)p.peak_rank);
    const double walk = 0.1 * frames + (1.0 + 0.05 * amps) * p.operations;
    const double shot = 0.25e-3 * frames + (0.3e-3 + 0.12e-3 * amps) * p.operations;
    return std::max(walk, (double)total / cus * shot);
}

// The shape in a batch of `total` shots, of which `shots` are this program's,
// and its estimated time (us): the least if the others are like it.  Teams beyond
// what a compute unit holds at once wait for each other; fewer leave compute
// units idle, and shots are then better spread over more teams (8 random
// programs of peak 8 with 1000 shots, in one team each 3.6 ms, 0.58 so).  Two team
// sizes, the larger alone for states in memory: each more is one more launch
// with an end of its own (512 Clifford+T programs of peak 4 to 16, 1000 shots
// each, all of 64 to 1024 threads: 766 us, 256 and 1024: 572, 1024 alone:
// 552, 512 alone: 735); smaller ones where the records leave no room.
// Negative: none.
inline double tree_batch_shape(const TreeProfile& p, uint64_t shots, uint64_t total, double cus, TreeShape& best) {
    double cost = -1.0;
    for (uint32_t threads : {1024u, 256u, 64u}) {
        if (cost >= 0.0 && threads == 64u) break;
        for (uint32_t chunk = threads; chunk >= 1; chunk /= 2) {
            if (chunk > 64 && chunk >= 2 * shots) continue;
            TreeShape s;
            if (!tree_team(p, threads, chunk, 0, s) || (cost >= 0.0 && s.global && threads < best.threads)) continue;
            if (chunk > 1 && s.elems > tree_room(p)) continue;
            const double part = std::max((double)threads / 1024.0, (double)s.lds / (double)kTreeCuLds);
            const double teams = std::ceil((double)shots / chunk) * ((double)total / (double)shots) / cus;  // a compute unit
            const double c = std::max(1.0, teams * part) * tree_team_us(p, s, std::clamp(teams, 1.0, 1.0 / part));
            if (cost < 0.0 || c < cost) {
                best = s;
                cost = c;
            }
        }
    }
    return cost;
}

// The programs of a batch that share their states, each with its shape (0
// threads: not).  From peak 7 on, and beyond 64 qubits, all that have a plan do;
// the others all or none, by their estimates together: a lane group for a few
// of them takes its whole walk beside the teams' (random programs of peak 6, 64
// with 1000 shots: 1.15 ms with three of them on lanes, 0.61 with none).  Where
// the device is full the estimate of the teams is low by 1.3 (peak 5, 256 random
// programs with 1000 shots: 1.5 ms on teams, 1.25 on lanes).
inline std::vector<TreeShape> tree_batch(const std::vector<const TreeProfile*>& progs, const std::vector<uint64_t>& shots,
                                         double cus, int mode) {
    std::vector<TreeShape> out(progs.size());
    if (mode == 0) return out;
    uint64_t total = 0;
    for (uint64_t n : shots) total += n;
    auto low = [&](const TreeProfile& p) { return mode == 1 && p.frame_words == 1 && p.peak_rank <= 6; };
    double teams = 0.0, lanes = 0.0;
    for (size_t i = 0; i < progs.size(); ++i) {
        const TreeProfile& p = *progs[i];
        if (!p.ok || shots[i] == 0) continue;
        TreeShape s;
        const double c = tree_batch_shape(p, shots[i], total, cus, s);
        if (c < 0.0) continue;
        out[i] = s;
        if (!low(p)) continue;
        teams += c * (double)shots[i];
        lanes += batch_lanes_us(p, total, cus) * (double)shots[i];
    }
    if (1.3 * teams > lanes)
        for (size_t i = 0; i < progs.size(); ++i)
            if (low(*progs[i])) out[i] = TreeShape();
    return out;
}

}  // namespace csvm
