"""The order of LDS accesses in a diagonal block with a panel pending (csrc/diag_schedule.h, which the kernel
takes its schedule from): whatever a wave touches in the first strip, no other wave may still be applying
the panel to it, or reading the panel's parts from under it; and in every strip each block has one wave, which
finds the rows that it needs there."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), 'pytorch-sso_amd', 'csrc')

PROGRAM = r'''
#include <cstdio>
#include "diag_schedule.h"
using namespace kfac;
int main() {
  for (int w = 0; w < PENDING_WAVES; ++w) printf("pending %d %d %d\n", w, pending_row(w), pending_col(w));
  for (int q = 0; q < 4; ++q) {
    for (int w = 0; w < DIAG_WAVES; ++w) printf("role %d %d %d\n", q, w, (int)(STRIP_ROLES[q] >> (5 * w)) & 31);
    for (int nq = q + 1; nq <= 4; ++nq)
      for (int h = 0; h < STRIP_HELPERS; ++h)
        helped_blocks(q, nq, h, [&](int i, int col) { printf("helped %d %d %d %d %d\n", q, nq, h, i, col); });
  }
  for (int col = 0; col < 8; ++col) printf("from %d %d\n", col, helped_from(col));
  printf("row0 %d\n", PENDING_ROW0);
}
'''


@pytest.fixture(scope='module')
def schedule(tmp_path_factory):
    d = tmp_path_factory.mktemp('schedule')
    (d / 'main.cpp').write_text(PROGRAM)
    subprocess.run(['g++', '-std=c++17', '-I', CSRC, str(d / 'main.cpp'), '-o', str(d / 'main')], check=True)
    rows = {}
    for line in subprocess.run([str(d / 'main')], check=True, capture_output=True, text=True).stdout.splitlines():
        kind, *values = line.split()
        rows.setdefault(kind, []).append(tuple(int(v) for v in values))
    return rows


def role(code):
    return ('lead', 0) if code == 1 else ('collect', code - 16) if code >= 16 else \
        ('follow', code - 8) if code >= 8 else ('help', code - 2) if code >= 2 else ('none', 0)


def test_the_panel_is_applied_to_every_block_once(schedule):
    assert sorted((i, j) for _, i, j in schedule['pending']) == [(i, j) for i in range(4) for j in range(i, 4)]


def test_roles_cover_every_strip(schedule):
    for q in range(4):
        roles = [role(code) for s, _, code in schedule['role'] if s == q]
        assert roles.count(('lead', 0)) == 1
        # the rest of the row panel, and the blocks of Z up to the strip's own
        assert sorted(c for kind, c in roles if kind == 'follow') == list(range(q + 1, 4)) + [4 + c for c in range(q + 1)]
        assert sorted(h for kind, h in roles if kind == 'help') == [0, 1, 2]
    for q in range(3):      # who collects a block for the next strip has it there
        now = {w: role(code) for s, w, code in schedule['role'] if s == q}
        then = {w: role(code) for s, w, code in schedule['role'] if s == q + 1}
        for w, (kind, c) in now.items():
            if kind == 'collect':
                assert then[w] == (('lead', 0) if c == q + 1 else ('follow', c))


def test_helped_blocks_are_the_rows_further_down(schedule):
    for q in range(4):
        for nq in range(q + 1, 5):
            got = sorted(r[3:] for r in schedule.get('helped', []) if r[:2] == (q, nq))
            want = [(i, j) for i in range(q + 2, nq) for j in list(range(i, nq)) + [4 + c for c in range(q + 1)]]
            assert got == sorted(want)


def touched(schedule, q, nq):
    """(wave, role, block) of every block of S or Z that a wave reads or writes in strip q of a block of nq strips.
    Collecting waves read finished rows of the strip only, behind their marks."""
    for s, w, code in schedule['role']:
        kind, c = role(code)
        if s != q:
            continue
        if kind == 'lead':
            yield w, kind, (q, q)
        elif kind == 'follow' and (c < nq if c < 4 else c - 4 <= q):
            yield w, kind, (q, c)
        elif kind == 'help' and q > 0:
            for r in schedule.get('helped', []):
                if r[:3] == (q - 1, nq, c) and r[3] == q + 1:
                    yield w, kind, r[3:]


@pytest.mark.parametrize('nq', [1, 2, 3, 4])
def test_no_access_of_the_first_strip_overtakes_the_pending_panel(schedule, nq):
    owner = {(i, j): w for w, i, j in schedule['pending']}
    row0 = schedule['row0'][0][0]
    blocks = list(touched(schedule, 0, nq))
    assert len(blocks) == nq + 1 and all(kind != 'help' for _, kind, _ in blocks)
    for w, _, (i, col) in blocks:
        # whose accesses have to be over: the block's owner's, or, where the panel's parts lie, everybody's
        before = {owner[i, col]} if col < 4 else set(owner.values()) if 32 * i + 31 >= row0 else set()
        assert before <= {w}, 'wave %d in block (%d, %d)' % (w, i, col)


@pytest.mark.parametrize('nq', [1, 2, 3, 4])
def test_helpers_take_what_the_strips_above_give_to_the_next_one(schedule, nq):
    """A helper of strip q: one block at most, of block row q + 1, which nobody else touches then; the strips that
    it takes from are above q, at most two, and all that give something to the block but strip q, which the
    block's own wave collects."""
    first = dict(schedule['from'])
    for q in range(nq):
        blocks = list(touched(schedule, q, nq))
        assert len(set(b for _, _, b in blocks)) == len(blocks) == len(set(w for w, _, _ in blocks))
        helped = sorted(b for _, kind, b in blocks if kind == 'help')
        want = [(q + 1, j) for j in list(range(q + 1, nq)) + [4 + c for c in range(q)]] if 0 < q < nq - 1 else []
        assert helped == want
        for i, col in helped:
            gives = [s for s in range(i) if col < 4 or s >= col - 4]
            assert gives == list(range(first[col], q + 1)) and 1 <= q - first[col] <= 2


def test_every_row_is_written_once(schedule):
    """Rows of strip q - 1, in sixteen pieces: in strip q the collecting waves have the pieces 4 (c - q - 1) + (0 ... 3);
    strip 3 has no such waves, but some without a block."""
    for q in (1, 2):
        columns = [role(code)[1] for s, _, code in schedule['role'] if s == q and role(code)[0] == 'collect']
        assert sorted(4 * (c - q - 1) + k for c in columns for k in range(4)) == list(range(16))
    last = [role(code)[0] for s, _, code in schedule['role'] if s == 3]
    assert 'collect' not in last and any(kind in ('help', 'none') for kind in last)


def test_the_kernel_takes_its_schedule_from_the_header():
    with open(os.path.join(CSRC, 'inverse.hip')) as f:
        text = f.read()
    block = text[text.index('void diag_block('):text.index('void potrf_diag_kernel')]
    for name in ('STRIP_ROLES', 'helped_blocks', 'helped_from', 'pending_row', 'pending_col', 'PENDING_WAVES',
                 'PENDING_ROW0'):
        assert name in block
