// svm_tree_args.h -- tables of the shared-state executor (svm_tree.h),
// produced by the host planner (svm_tree_plan.h).
#pragma once

#include <stdint.h>

namespace csvm {

// The shots' classical part is linear over GF(2): every record, detector and
// observable bit, and every bit the walk has to read (whether a shot parts
// from its node, a post-selection parity, the sign of an expectation value),
// is a constant plus the sum of some of the shot's random bits.  A shot
// therefore keeps these bits themselves (its "response"), starting from the
// constants, and each random bit that comes up 1 adds the row of bits it
// flips.  The Pauli frame and all opcodes that only move it are gone.
//
// Response: words of 32 bits -- measurement records, detectors, observables,
// then the bits that are read -- each section starting on a word.
// `dense` holds whole responses: number 0 the constants, the others sets of
// bits to keep.  A row is what one random bit flips, few of the words: a list
// of (word << 6, mask), the masks nonzero.  `rows` is made of units of four
// such entries; the rows that an opcode names lie one after another, all of
// axis_2 units, filled up with zeros.
//
// Opcodes (payload word 1 unless stated; a bit is word * 32 + position; a
// row is named by its first unit):
//   kLpRandom      axis_1 coin flips, rows from i1 on
//   kLpNoise       the noise sites [i0, i1)
//   kLpReadout     axis_1 readout-noise entries from i0 on, rows from i1 on
//   kLpPostselect  the shot is discarded if bit i0 is set, keeping the bits
//                  of response i1 of `dense`
//   kLpCoin        forced coin flip of record i0, row i1
//   kLpStatic      forced: record i0 has to equal its response bit
//   kTreeChoice    the shots of a node part by the `reserved` bits from i0 on
//                  (one word); payload word 2 = their place in the choice word
//   kTreeMeas      active measurement into record i0, row i1 flipped by
//                  outcome 1 (reserved bit 0: forced)
//   kTreePass      a pass with no per-shot part
//   kTreeNode      U2 (reserved 2) or U4 (reserved 4) node i0: its frame
//                  state from the `reserved` bits at bit i1; payload word 2 =
//                  first of as many rows, one per bit of the state it leaves
//   kTreeEv        EXP_VAL: output i0, sign bit i1, payload word 2 = kind (0:
//                  computed, 1: the value is 0, 2: it is +-1 by the sign)
// kTreeMeas, kTreePass and the computed kTreeEv each run the next pass of
// the plan: the program is straight-line, so passes run in table order.
// The walk reads one instruction ahead: a spare one follows the last.
constexpr uint32_t kLpRandom = 0xD0;
constexpr uint32_t kLpNoise = 0xD1;
constexpr uint32_t kLpReadout = 0xD2;
constexpr uint32_t kLpPostselect = 0xD3;
constexpr uint32_t kLpCoin = 0xD4;
constexpr uint32_t kLpStatic = 0xD5;
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
constexpr uint32_t kTreeMaxWords = 512;  // of a shot's response

// A noise site: its channels [first, first + n) and its cumulative hazard.
struct TreeSite {
    uint32_t first, n;
    double hazard;
};
// A channel: the running sum of its site's channel probabilities, and the
// row it adds: entries [first, first + n), first even.
struct TreeChan {
    double cum;
    uint32_t first, n;
};

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

struct TreeStage {  // the running pass's expansion products
    double tab[1u << kTreeMaxExpand][2];
};
constexpr uint32_t kTreeParts = 128;  // partial sums of a pass with several per node

// LDS of one team of `threads` threads and at most `chunk` shots: per-wave
// response columns (64 x 4 B a word; with k-fault sampling also the fault
// lists), two node tables (source node, choice word), per-node
// sums, partial sums, two key bitmaps (and the rescale flag), the stage.
constexpr uint32_t tree_flag_words(uint32_t chunk) { return (chunk + 1u) / 2u + 2u; }
constexpr uint32_t tree_lds_bytes(uint32_t threads, uint32_t chunk, uint32_t lane_words) {
    uint32_t b = (threads >> 6) * lane_words * 256u;
    b += (16u * chunk + 15u) / 16u * 16u;  // 4 x u32 tables
    b += 16u * chunk + 16u * kTreeParts;
    b += (8u * tree_flag_words(chunk) + 15u) / 16u * 16u;
    return b + (uint32_t)sizeof(TreeStage);
}

}  // namespace csvm
