// The plan of a preconditioning (precond.hip): which tiles each step of its products has, into which pieces
// their reductions are cut, and how much room the pieces take.  Plain arithmetic:
// tests/test_precond_plan.py compiles this file and checks that the room holds the pieces of every call.
// (The kernels count their tiles by the same functions.  Those are `inline`: as constexpr functions only they were
// called, not inlined, and AlexNet's layers took 14060 instead of 13830 us a step.)
#pragma once
#include <vector>

#include "common.h"

namespace kfac {

// what the operands of a layer are: triangular factors (else explicit inverses), R's in two halves
enum { L_FACTOR = 1, R_FACTOR = 2, R_HALVES = 4 };

constexpr int PLAN_TILE = 128;

// A reduction against a triangular operand of T blocks is up to T blocks long, and a launch
// lasts at least as long as its longest tile: a 4608-deep tile is 150 MFLOP on ONE compute
// unit.  Where that is longer than the launch would take if its work were spread evenly
// (few layers, or few tiles: the driver decides per product), the reductions are cut into
// pieces of at most `pb` blocks, each a work item of the same launch that stores a raw
// partial tile; a second, short launch adds the pieces of every cut tile up in order and
// applies the epilogue (precond_finish_kernel).  Piece j exists for the tiles whose
// reduction is longer than j * pb blocks: tfast - j * pb values of `fast`.  pb == 0: no
// reduction is cut.
enum { PART_A = 0, COUPLING = 1, PART_B = 2, STEPS = 3 };
constexpr int PRODUCTS = 4;
__host__ __device__ inline int half_of(int T) { return T >> 1; }     // blocks of the first half

// which of the T tiles along the reduction a part holds (`grows`: the reduction gets longer with the
// tile index, so that the first half comes first); their reductions start or end where the part does
struct TileRange {
  int first, count;
};
__host__ __device__ inline TileRange part_tiles(int T, bool halves, bool grows, int part) {
  if (!halves) return part == PART_A ? TileRange{0, T} : TileRange{0, 0};
  const int h = half_of(T);
  return (part == PART_A) == grows ? TileRange{0, h} : TileRange{h, T - h};
}

// pieces of a reduction of `blocks` 128-blocks cut at `pb` blocks (pb <= 0: not cut)
__host__ __device__ inline int piece_count(int blocks, int pb) { return pb > 0 ? (blocks + pb - 1) / pb : 1; }

// work items of a layer in one product: tiles x pieces
__host__ __device__ inline int piece_items(int tslow, int tfast, bool tri, int pb) {
  if (pb <= 0) return tslow * tfast;
  if (!tri) return tslow * tfast * piece_count(tfast, pb);    // dense: all reductions tfast blocks
  int n = 0;
  for (int j = 0; j * pb < tfast; ++j) n += tslow * (tfast - j * pb);
  return n;
}

// The couplings of the second (`product` 1) and third (2) product: the tiles of PART_B's input, `slow`
// over dG and `fast` over its blocks of dA; reductions over all of PART_A, `depth` blocks.
struct CouplingShape {
  int first, count;              // blocks of PART_B
  int kfirst, depth;             // of PART_A
};
__host__ __device__ inline CouplingShape coupling_shape(int product, int ta, int flags) {
  const bool grows = product == 1;
  const TileRange a = part_tiles(ta, true, grows, PART_A), b = part_tiles(ta, true, grows, PART_B);
  return CouplingShape{b.first, flags & R_HALVES ? b.count : 0, a.first, a.count};
}

// what a layer does in one step of a product: `tiles` tiles with reductions of up to `longest` blocks
// (tri: of 1 to `longest`, with `tslow` of each length), `work` blocks in all
struct StepShape {
  int tiles, longest, tslow;
  bool tri;
  long work;
};
inline StepShape step_shape(int product, int step, int dG, int dA, int flags, bool sample) {
  const int ta = cdiv(dA, PLAN_TILE), tg = cdiv(dG, PLAN_TILE);
  const bool over_g = product == 0 || product == 3;
  const bool tri = sample || (flags & (over_g ? L_FACTOR : R_FACTOR));
  if ((product >= 2 && (!tri || sample)) || (sample && step != PART_A)) return StepShape{0, 0, 1, false, 0};
  const bool halves = !over_g && (flags & R_HALVES);
  if (step == COUPLING) {
    const CouplingShape cs = coupling_shape(product, ta, flags);
    return halves ? StepShape{tg * cs.count, cs.depth, tg, false, (long)tg * cs.count * cs.depth}
                  : StepShape{0, 0, 1, false, 0};
  }
  const int count = part_tiles(over_g ? tg : ta, halves, product < 2, step).count;
  const int tslow = over_g ? ta : tg;
  return StepShape{tslow * count, count, tslow, tri,
                   tri ? (long)tslow * count * (count + 1) / 2 : (long)tslow * count * count};
}

// Piece size of each step of each product from the shape of its launch.  flags == nullptr: every side
// of every layer is a triangular factor (what the scratch is sized for, but for halves).
typedef int PieceSizes[PRODUCTS][STEPS];
inline void plan_pieces(int layers, const int* dG, const int* dA, const int* flags, PieceSizes& pbs,
                        bool sample = false) {
  for (int product = 0; product < PRODUCTS; ++product)
    for (int step = 0; step < STEPS; ++step) {
      long work = 0;
      int longest = 0;
      for (int l = 0; l < layers; ++l) {
        const StepShape sh = step_shape(product, step, dG[l], dA[l], flags ? flags[l] : L_FACTOR | R_FACTOR,
                                        sample);
        work += sh.work;
        longest = std::max(longest, sh.longest);
      }
      pbs[product][step] = piece_blocks(work, longest);
    }
}

// The sizes that a call uses, under the plan `room` that the scratch was sized for (the query assumed that
// every side is a triangular factor): pieces as large as that plan's, at least, and none where it left no room.
inline void call_pieces(int layers, const int* dG, const int* dA, const int* flags, const PieceSizes& room,
                        PieceSizes& pbs, bool sample) {
  plan_pieces(layers, dG, dA, flags, pbs, sample);
  for (int product = 0; product < PRODUCTS; ++product)
    for (int step = 0; step < STEPS; ++step) {
      int& pb = pbs[product][step];
      pb = pb > 0 && room[product][step] > 0 ? std::max(pb, room[product][step]) : 0;
    }
}

// tiles of the piece area of a layer under the piece sizes `pbs`: room for the pieces of
// the longest reduction, for every tile
inline size_t piece_tiles(int dG, int dA, int flags, const PieceSizes& pbs) {
  size_t most = 0;
  for (int product = 0; product < PRODUCTS; ++product)
    for (int step = 0; step < STEPS; ++step) {
      const StepShape sh = step_shape(product, step, dG, dA, flags, false);
      const int pieces = piece_count(sh.longest, pbs[product][step]);
      if (pieces > 1) most = std::max(most, (size_t)sh.tiles * pieces);
    }
  return most;
}

// The same as floats, for a layer that the query was told `room` of (L_FACTOR etc.).  A layer in halves has room for
// whole operands as well: the query does not know which operands are factors, and where R is not one, its
// products run over all of it (dG = 64, dA = 9216: 1080 tiles, in halves 432).
inline size_t piece_floats(int dG, int dA, int room, const PieceSizes& pbs) {
  size_t tiles = piece_tiles(dG, dA, room, pbs);
  if (room & R_HALVES) tiles = std::max(tiles, piece_tiles(dG, dA, room & ~R_HALVES, pbs));
  return tiles * (PLAN_TILE * PLAN_TILE);
}

// what is in halves, as plan_pieces wants it (a matrix of one block has none)
inline std::vector<int> halves_room(int layers, const int* dA, const int* a_halves) {
  std::vector<int> flags(layers, L_FACTOR | R_FACTOR);
  for (int l = 0; l < layers; ++l)
    if (a_halves[l] && half_of(cdiv(dA[l], PLAN_TILE)) > 0) flags[l] |= R_HALVES;
  return flags;
}

// what the operands of a call are (NULL: all factors), with the halves of `room` (NULL: none) where R is a factor
inline std::vector<int> operand_flags(int layers, const int* g_factored, const int* a_factored, const int* room) {
  std::vector<int> flags(layers);
  for (int l = 0; l < layers; ++l) {
    const bool a = !a_factored || a_factored[l];
    flags[l] = ((!g_factored || g_factored[l]) ? L_FACTOR : 0) | (a ? R_FACTOR : 0) |
               (a && room ? room[l] & R_HALVES : 0);
  }
  return flags;
}

}  // namespace kfac
