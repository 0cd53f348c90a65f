// Who does what in a diagonal block of the Cholesky (diag_block of inverse.hip), and the order in which a pending
// panel is applied to it.  Constants and constant expressions only: tests/test_diag_schedule.py compiles this
// file for the host and checks that no wave touches what another one may still be using.
#pragma once

namespace kfac {

// Which wave does what in strip q.  Block columns: 1-3 of S (the row panel), 4-7 = 0-3 of Z.
//   LEAD: the leaf;  FOLLOW c: the block of column c;  COLLECT c: what strip q takes from the block
//   of column c in strip q+1, which that wave then follows, or leads, with;  HELP: the rest.
// A SIMD has the waves s, s+4, s+8 and issues one instruction at a time to its matrix core or its
// vector unit; of a step, the leading wave takes it 160 cycles, a following one 90, a collecting
// one 70, and a helper 1400 cycles for a block.  So the leading wave has no following one beside
// it, and every SIMD has about the same to do:
//   SIMD      0               1                     2                    3
//   strip 0   lead, C4, H     F1, C1, H             F2, C2, H            F3, C3, F4
//   strip 1   C4, F4, F5      lead, C5, H (1)       C2, F2, H (2)        C3, F3, H (2 blocks)
//   strip 2   F4, C4, C5      F6, F5, C6            lead, H, H (2)       F3, C3, H (1)
//   strip 3   F4, F5          F6, H                 F7, H, H             lead
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
    StripRoles().set(0, ROLE_LEAD).set(4, ROLE_COLLECT, 4).set(8, ROLE_HELP, 0)
        .set(1, ROLE_FOLLOW, 1).set(5, ROLE_COLLECT, 1).set(9, ROLE_HELP, 1)
        .set(2, ROLE_FOLLOW, 2).set(10, ROLE_COLLECT, 2).set(6, ROLE_HELP, 2)
        .set(3, ROLE_FOLLOW, 3).set(7, ROLE_COLLECT, 3).set(11, ROLE_FOLLOW, 4).bits,
    StripRoles().set(0, ROLE_COLLECT, 4).set(4, ROLE_FOLLOW, 4).set(8, ROLE_FOLLOW, 5)
        .set(5, ROLE_LEAD).set(9, ROLE_COLLECT, 5).set(1, ROLE_HELP, 0)
        .set(2, ROLE_COLLECT, 2).set(10, ROLE_FOLLOW, 2).set(6, ROLE_HELP, 1)
        .set(3, ROLE_COLLECT, 3).set(7, ROLE_FOLLOW, 3).set(11, ROLE_HELP, 2).bits,
    StripRoles().set(0, ROLE_FOLLOW, 4).set(4, ROLE_COLLECT, 4).set(8, ROLE_COLLECT, 5)
        .set(5, ROLE_FOLLOW, 6).set(9, ROLE_FOLLOW, 5).set(1, ROLE_COLLECT, 6)
        .set(2, ROLE_LEAD).set(6, ROLE_HELP, 0).set(10, ROLE_HELP, 1)
        .set(3, ROLE_FOLLOW, 3).set(7, ROLE_COLLECT, 3).set(11, ROLE_HELP, 2).bits,
    StripRoles().set(4, ROLE_FOLLOW, 4).set(8, ROLE_FOLLOW, 5)
        .set(1, ROLE_FOLLOW, 6).set(5, ROLE_HELP, 0)
        .set(6, ROLE_FOLLOW, 7).set(2, ROLE_HELP, 1).set(10, ROLE_HELP, 2)
        .set(7, ROLE_LEAD).bits};

// The blocks that strip q changes in the rows further down, of a block of nq strips:  (i, i), (i, i+1), ...
// of S and (i, 0), ... (i, q) of Z for the block rows i > q + 1; at most five, two to a helper.
template <class F>
constexpr void helped_blocks(int q, int nq, int helper, F&& take) {
  int k = 0;
  for (int i = q + 2; i < nq; ++i)
    for (int b = 0; b < nq - i + q + 1; ++b, ++k)
      if (k % STRIP_HELPERS == helper) take(i, b < nq - i ? i + b : 4 + b - (nq - i));
}

// A pending panel is applied by ten waves, a 32x32 block of S each, from parts that lie in the rows of Z from
// PENDING_ROW0 on.  The waves 0-3 have the blocks that they begin strip 0 with, and go on without waiting for
// anybody.  Nothing of the others' is read or written in strip 0 (the blocks of the rows below belong to strip 1,
// behind a barrier) but by its helpers: they change S(2,2), S(2,3), S(3,3), which the waves 7-9 update, and
// write Z(2,0), Z(3,0), over parts that any wave may still be reading.  What they wait for otherwise, the rows
// of strip 0, does not depend on the waves 1 and 4-9.  So each wave leaves a mark when it is done with the
// panel, behind its last access to S and to the parts, and a helper of strip 0 waits for all of them before it
// touches its first block.
constexpr int PENDING_WAVES = 10, PENDING_ROW0 = 32;
constexpr int pending_row(int wave) { return (int)(0x3221110000ull >> (4 * wave)) & 3; }
constexpr int pending_col(int wave) { return (int)(0x3323213210ull >> (4 * wave)) & 3; }
constexpr bool helper_awaits_pending(int q) { return q == 0; }

}  // namespace kfac
