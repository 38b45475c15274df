// svm_tree_args.h -- tables of the shared-state executor (svm_tree.h),
// produced by the host planner (svm_tree_plan.h).
#pragma once

#include <stdint.h>

namespace csvm {

// Tree-bytecode opcodes (below the lane superinstructions, above the
// reference's range).
//   kTreeChoice  the shots of a node part by frame bits that the amplitudes
//                depend on: reserved = how many bits (1: p_x of axis_1; 2:
//                p_x, p_z of axis_1; 4: those of axis_1, then of axis_2),
//                payload word 1 = their place in the node's choice word
//   kTreeMeas    active measurement of axis_1 (reserved bit 0: interfere,
//                else diagonal; bit 1: forced); payload word 1 = record
//                index
//   kTreePass    a pass with no per-shot part
//   kTreeNode    the frame of a U2 (reserved 0) or U4 (reserved 1)
//                node, payload word 1 = node index
//   kTreeEv      EXP_VAL: payload word 1 = mask index | output index << 32,
//                word 2 = kind (0: computed, 1: the value is 0, 2: it is +-1
//                by the sign alone)
// kTreeMeas, kTreePass and the computed kTreeEv each run the next pass of
// the plan: the program is straight-line, so passes run in table order.
constexpr uint32_t kTreeChoice = 0xE0;
constexpr uint32_t kTreeMeas = 0xE1;
constexpr uint32_t kTreePass = 0xE2;
constexpr uint32_t kTreeNode = 0xE3;
constexpr uint32_t kTreeEv = 0xE4;

// What a pass does with the entries it computes.  Every type but TREE_U4
// and TREE_EV works on the pairs (i, 0), (i, 1), i < 2^(r-1), of coordinate
// indices whose top bit is the pair's.
enum : uint32_t {
    TREE_COPY = 0,       // write both
    TREE_DIAG = 1,       // write both (the states of outcomes 0 and 1), sum |.|^2 of each
    TREE_INTERFERE = 2,  // write (p + q) / sqrt 2 and (p - q) / sqrt 2, sum |p + q|^2 and |p - q|^2
    TREE_H = 3,          // write (p + q) / sqrt 2 and (p - q) / sqrt 2
    TREE_U2 = 4,         // write the node's 2x2 of (p, q)
    TREE_U4 = 5,         // write the node's 4x4 of the quad of the top two bits
    TREE_EV = 6,         // sum the EXP_VAL numerator and norm over pairs (y, y ^ xa)
    TREE_EV0 = 7         // the same for a string without X (each entry on its own)
};

constexpr uint32_t kTreeMaxExpand = 5;   // pending expansions a pass reads through
constexpr uint32_t kTreeMaxGen = 31;     // general phases of a pass
constexpr uint32_t kTreeMaxChoice = 32;  // bits of a node's choice word
constexpr uint32_t kTreeMaxRank = 26;

// General phase of a pass: the entry is multiplied by (pr, pi), by its
// conjugate where the node's choice bit is set (choice < 0: never).
struct TreePhase {
    int32_t choice;
    uint32_t pad;
    double pr, pi;
};

// One pass over the stored amplitudes of every node.  A coordinate index y
// (r bits) has four words, each the XOR of that array's entries over the set
// bits of y (index words are byte offsets: times 16):
//   cols  the stored index x the entry comes from: its low r0 bits name the
//         stored entry, the m bits above them the pending expansions (phase
//         ez[b], conjugated where the node's choice bit is set; ez_tab: the
//         products for every value of the m bits when no choice is involved)
//   colg  general phase j (table entries gen_off + j, applied in order)
//         multiplies the entry where bit j is set
//   colo  (pair bits have none) the index of the pair in the written state:
//         entry colo, and colo + 2^(r-1); TREE_U4: colo + c 2^(r-2), c < 4
//   cols_s  signs of the pair's upper entry relative to its lower one: bit
//         31, XOR sign0's (TREE_U4: bits 31, 30, 29 for corners 1, 2, 3)
// The upper entry also turns by i where bit 31 of `quarter` is set (TREE_U4:
// the corners' bits).  Phases common to a pair are not applied: the planner
// carries them on to the next pass.
// The first 160 words are read by each wavefront's lanes.
struct TreePass {
    uint32_t type;
    uint32_t r0, m, r;
    uint32_t quarter;
    uint32_t ngen, gen_off;
    uint32_t sign0;
    uint32_t ez_choices;  // some expansion's phase depends on the choice word
    uint32_t reset;       // the pass consumes every pending choice
    uint32_t node;        // TREE_U2 / TREE_U4
    uint32_t choice;      // their place in the choice word
    uint32_t evz;         // TREE_EV*: Z mask on coordinate indices
    uint32_t ev_imag;     // TREE_EV*: the phase i^|x & z| is imaginary
    int32_t ev_sign;      // its sign (+-1)
    int32_t ez_choice[kTreeMaxExpand];
    uint32_t pad[12];
    uint32_t cols[32], colo[32], cols_s[32], colg[32];
    double ez[kTreeMaxExpand][2];
    double ez_tab[1u << kTreeMaxExpand][2];
};

}  // namespace csvm
