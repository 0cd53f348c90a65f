// Who does what in a diagonal block of the Cholesky (diag_block of inverse.hip), and the order in which a pending
// panel is applied to it.  Constants and constant expressions only: tests/test_diag_schedule.py compiles this
// file for the host and checks that no wave touches what another one may still be using.
#pragma once

namespace kfac {

// Which wave does what in strip q.  Block columns: 1-3 of S (the row panel), 4-7 = 0-3 of Z.
//   LEAD: the leaf;  FOLLOW c: the block of column c;  COLLECT c: what strip q takes from the block
//   of column c in strip q+1, which that wave then follows, or leads, with;  HELP: the rest.
// What a helper does is not what strip q is about: it takes what the strips above q give to a block of strip
// q+1, whose rows are all there, so that it waits for nobody and nobody for it (in strip q itself, behind the
// last rows of the followers, it was what the strip ended with: 0.7 to 1.6 us each).
// A SIMD has the waves s, s+4, s+8 and issues one instruction at a time to its matrix core or its
// vector unit; of a step, the leading wave takes it 160 cycles, a following one 90, a collecting
// one 70, and a helper 1400 cycles for a block and strip.  The leading wave is slowed by whatever else its SIMD
// does, by the bursts of a helper most (an idle SIMD 1.5 us a strip, with a collecting and a following wave or a
// helper of one strip 2.0, with two helpers 2.6), and starts on a SIMD of two waves with a pending block:
//   SIMD      0                    1                2                    3
//   strip 0   F2, C2               F1, C1           lead, C4             F3, C3, F4
//   strip 1   C2, F2, H (1 strip)  lead, C5, F5     C4, F4, H (1)        C3, F3, H (1)
//   strip 2   lead, C5, H (1)      F6, F5, C6       F4, C4, H (2)        F3, C3, H (2)
//   strip 3   F5                   F6               F4, F7               lead
enum { ROLE_NONE = 0, ROLE_LEAD = 1, ROLE_FOLLOW = 2, ROLE_COLLECT = 3, ROLE_HELP = 4 };
constexpr int DIAG_WAVES = 12;
constexpr int STRIP_HELPERS = 3;
struct StripRoles {
  unsigned long long bits = 0;      // 5 bits a wave
  static constexpr unsigned long long code(int kind, int c) {
    return kind == ROLE_LEAD ? 1 : kind == ROLE_HELP ? 2 + c : kind == ROLE_FOLLOW ? 8 + c
           : kind == ROLE_COLLECT ? 16 + c : 0;
  }
  constexpr StripRoles& set(int wave, int kind, int c = 0) {
    bits |= code(kind, c) << (5 * wave);
    return *this;
  }
};
constexpr unsigned long long STRIP_ROLES[4] = {
    StripRoles().set(0, ROLE_FOLLOW, 2).set(4, ROLE_HELP, 2).set(8, ROLE_COLLECT, 2)
        .set(1, ROLE_FOLLOW, 1).set(5, ROLE_COLLECT, 1).set(9, ROLE_HELP, 1)
        .set(2, ROLE_LEAD).set(6, ROLE_COLLECT, 4).set(10, ROLE_HELP, 0)
        .set(3, ROLE_FOLLOW, 3).set(7, ROLE_COLLECT, 3).set(11, ROLE_FOLLOW, 4).bits,
    StripRoles().set(0, ROLE_COLLECT, 2).set(4, ROLE_HELP, 1).set(8, ROLE_FOLLOW, 2)
        .set(1, ROLE_FOLLOW, 5).set(5, ROLE_LEAD).set(9, ROLE_COLLECT, 5)
        .set(2, ROLE_COLLECT, 4).set(6, ROLE_FOLLOW, 4).set(10, ROLE_HELP, 2)
        .set(3, ROLE_COLLECT, 3).set(7, ROLE_FOLLOW, 3).set(11, ROLE_HELP, 0).bits,
    StripRoles().set(0, ROLE_LEAD).set(4, ROLE_COLLECT, 5).set(8, ROLE_HELP, 2)
        .set(1, ROLE_COLLECT, 6).set(5, ROLE_FOLLOW, 6).set(9, ROLE_FOLLOW, 5)
        .set(2, ROLE_FOLLOW, 4).set(6, ROLE_COLLECT, 4).set(10, ROLE_HELP, 0)
        .set(3, ROLE_FOLLOW, 3).set(7, ROLE_COLLECT, 3).set(11, ROLE_HELP, 1).bits,
    StripRoles().set(4, ROLE_FOLLOW, 5).set(1, ROLE_FOLLOW, 6).set(5, ROLE_HELP, 1)
        .set(9, ROLE_HELP, 2).set(2, ROLE_FOLLOW, 7).set(6, ROLE_FOLLOW, 4)
        .set(10, ROLE_HELP, 0).set(7, ROLE_LEAD).bits};

// The blocks that strip q changes in the rows further down, of a block of nq strips:  (i, i), (i, i+1), ...
// of S and (i, 0), ... (i, q) of Z for the block rows i > q + 1; at most five, and at most three of a block
// row, one to a helper.
template <class F>
constexpr void helped_blocks(int q, int nq, int helper, F&& take) {
  int k = 0;
  for (int i = q + 2; i < nq; ++i)
    for (int b = 0; b < nq - i + q + 1; ++b, ++k)
      if (k % STRIP_HELPERS == helper) take(i, b < nq - i ? i + b : 4 + b - (nq - i));
}

// The first strip that gives something to a block of block column `col` further down: the rows of S begin with
// strip 0, those of block column 4 + c of Z with strip c.  A helper of strip q takes the strips from there to q - 1.
constexpr int helped_from(int col) { return col < 4 ? 0 : col - 4; }

// A pending panel is applied by ten waves, a 32x32 block of S each, from parts that lie in the rows of Z from
// PENDING_ROW0 on.  The waves 0-3 have the blocks that they begin strip 0 with, and go on without waiting for
// anybody.  Nothing of the others' is read or written in strip 0: its collecting waves read its own rows, its helpers
// have no block yet, and the blocks of the rows below, also those of Z that lie over the parts, belong to the
// strips behind the barrier that ends strip 0.
constexpr int PENDING_WAVES = 10, PENDING_ROW0 = 32;
constexpr int pending_row(int wave) { return (int)(0x3221110000ull >> (4 * wave)) & 3; }
constexpr int pending_col(int wave) { return (int)(0x3321233012ull >> (4 * wave)) & 3; }

}  // namespace kfac
