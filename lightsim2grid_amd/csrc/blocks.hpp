// Block form of the factorisation plan: the unknowns of a bus (Va, and Vm of a PQ bus) are
// eliminated together as one 1 x 1 or 2 x 2 block.
//
// One block product replaces up to 8 scalar ones, and the dependency chains count buses instead of
// unknowns: on the 2000-bus grid 28 474 products in 33 levels where the scalar schedule has 136 790
// in 53 (10 000 buses: 214 561 in 71 against 834 922 in 82). The pattern is the exact one of the
// static elimination (L and U apart), so the reference slack's row takes no part where it is zero.
//
// Values are stored as pairs (2 consecutive numbers of one instance). A factor block (i, k) of L has
// one pair per row of bus i: (L(r, 0), L(r, 1)) over the columns of bus k. A block (k, j) of U has one
// pair per column of bus j: (U(0, c), U(1, c)) over the rows of bus k. The inner dimension is always
// padded to 2 with zeros, so a product L D U needs no test of a block's size. A diagonal block takes
// two row pairs and ends as the inverse of its pivot block; a right-hand side / solution entry of a bus
// is one pair. The tail of the elimination order is factored as one dense matrix.
#pragma once

#include <cstdint>
#include <vector>

#include "analysis.hpp"

namespace pfgpu {

// Target word of a block: where it is stored and how.
constexpr int kBlkAddrBits = 20;                   // pair index
constexpr int kBlkAddrMask = (1 << kBlkAddrBits) - 1;
constexpr int kBlkIn2 = 1 << 20;                   // the pairs' second numbers are in use
constexpr int kBlkTwo = 1 << 21;                   // the block has a second pair (a pivot always)
constexpr int kBlkCols = 1 << 22;                  // stored by columns (U, right-hand sides), else by rows
constexpr int kBlkInv = 1 << 23;                   // a pivot: its inverse is stored
constexpr int kBlkAssign = 1 << 24;                // fill-in: the target takes -sum
// and in the units of the lane streams
constexpr int kBlkLead = 1 << 25;                  // this lane writes the target
constexpr int kBlkTeamShift = 26;                  // 3 bits: log2 of the team, the same for the whole wave
constexpr int kBlkEnd = 1 << 29;                   // last unit of a task (whole wave)
constexpr int kBlkLevel = 1 << 30;                 // last unit of the wave's level
constexpr int kBlkWide = (int)(1u << 31);          // the block of U has two columns (backward); an operand of the
                                                   // wave lies outside LDS (factor)

// Unknowns of the dense tail at most: a wave factors it in registers, a column to a register and a row to
// a lane (nr_block_kernel.hpp), which at 1024 lanes leaves room for 48 columns of FP64. (The 10 000-bus grid's
// top chain has 88 unknowns: the 40 below the tail take 20 levels more, as long as the 40 took in a tail of 16
// waves.)
constexpr int kMaxTail = 48;

struct BlockPlan {
    int n = 0, m = 0;        // buses, unknowns of the dense tail
    int zpair = 0;           // two pairs that always hold zeros (0 and 1)
    int fixed_pairs = 2;     // the pairs below lie in LDS in every launch: the zeros, the tail's places
    int npairs = 0;          // value pairs of one instance, one pad pair at the end included
    int nlev = 0, nblev = 0;
    // per bus: the pair of its right-hand side (P, Q) and solution (dVa, dVm), kBlkIn2: two of them;
    // -1: no unknown. slack_x: the pair whose solution is the slack_absorbed step (of the reference
    // slack's bus), -1 without one
    std::vector<int> bus_y;
    int slack_x = -1, slack_bus = -1;
    // where the dense phase finds its matrix: per entry, row-major [m][m + 1], the number's place (2 pair +
    // component); column m is the right-hand side, which receives the solution
    std::vector<int> tail_src;
    // where blocks are stored, in the order of the pairs: first pair, pairs, accesses, whether it is empty while J
    // is assembled
    struct Place {
        int at, size;
        long long acc;
        bool fill;
    };
    std::vector<Place> places;
    std::vector<char> second;   // per pair: the second one of a block (npairs + 1 entries)
    // Assembly of F and J by Ybus rows (the buses with unknowns), longest first: per row {bus, its pair
    // word (bus_y), CSC position and target word of the diagonal entry}; the other entries as jagged
    // diagonals, entry k of row i at jd_ptr[k] + i: {column bus, target word (-1: no unknown there)} and
    // CSC position. J indices per entry and diagonal: dP/dVa, dQ/dVa, dP/dVm, dQ/dVm (-1: none).
    std::vector<int> rows, row_len, jd_ptr, jd, jd_pos, jd_jidx, row_jidx;
    // constant blocks: target word, values (00, 01, 10, 11), their J indices in the same order
    std::vector<int> jc_dst, jc_jidx;
    std::vector<double> jc_val;
    int fill_at = 0;  // pairs from here on hold no value while J is assembled (order kByLife), else npairs
    // factor + forward tasks by level: {target word, product begin, product end}; products {l, u, d};
    // backward tasks by level: {solution pair, begin, end, pair of the inverse pivot}; products
    // {u, x, 1 if the block has two columns}
    std::vector<int> f_lvl, tasks, prods, b_lvl, btasks, bprods;
};

// Whether J has the block form: its pivots on its own diagonal, and few enough values for the words.
bool has_block_form(const JPattern& J);
bool block_plan_fits(const BlockPlan& P);
// Order of the value pairs: by decreasing accesses (launches that spill keep the most used ones in LDS), or
// those in use while J is assembled first (launches with all of them in LDS can hold V in the rest then).
enum BlockOrder { kByUse = 0, kByLife = 1 };
// perm: the bus-block elimination order of J (column_order)
BlockPlan build_block_plan(const YbusPattern& Y, const JPattern& J, const std::vector<int>& perm, BlockOrder order = kByUse);
// a plan in order kByUse, in order kByLife
BlockPlan by_life(BlockPlan P);

// Pairs in LDS of a launch with room for `room` of an instance's: all of them, or as many as end between two
// blocks.
int lds_pairs(const BlockPlan& P, size_t room);

// Unit streams of the block plan for one launch shape: G interleaved instances, `waves` waves per
// workgroup, values of fsize bytes, the first nlds pairs in LDS. Each wave has a stream of its own of
// units of 64 lanes x 4 ints, one product per lane and unit, in level order:
//   factor    {l, u, d, word}   byte offsets of the operands (of instance 0), target word and control
//   backward  {u, x, d, word}   d: the task's inverse pivot, in its last unit
// A task's products are dealt to a team of 2^t lanes (t uniform over the wave), its last lane the
// leader; every lane of the wave walks the same number of units per task. Products that a lane lacks
// read the zero pairs. `mask`: per wave, one bit per level at which it has units.
struct BlockStreams {
    std::vector<int> fs, bs;            // units of all waves, wave after wave
    std::vector<int> f_at, b_at;        // first unit of each wave
    std::vector<uint64_t> f_mask, b_mask;  // [wave][words]
    int f_words = 1, b_words = 1;
};
constexpr int kBlkAhead = 4;  // units that a wave loads ahead; twice as many of padding end its stream
BlockStreams build_block_streams(const BlockPlan& P, int G, int waves, int fsize, int nlds);

}  // namespace pfgpu
