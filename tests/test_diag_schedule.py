"""The order of LDS accesses in a diagonal block with a panel pending (csrc/diag_schedule.h, which the kernel
takes its schedule from): whatever a wave touches in the first strip, the waves that may still be applying
the panel to it, or reading the panel's parts from under it, are waited for."""
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
    printf("awaits %d %d\n", q, (int)helper_awaits_pending(q));
  }
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


@pytest.mark.parametrize('nq', [1, 2, 3, 4])
def test_no_access_of_the_first_strip_overtakes_the_pending_panel(schedule, nq):
    owner = {(i, j): w for w, i, j in schedule['pending']}
    row0 = schedule['row0'][0][0]
    roles = {w: role(code) for s, w, code in schedule['role'] if s == 0}
    awaits = dict(schedule['awaits'])[0]
    for w, (kind, c) in roles.items():
        if kind == 'lead' or (kind == 'follow' and 0 < c < min(nq, 4)):
            touched = [(0, c)]
        elif kind == 'follow' and c == 4:
            touched = [(0, 4)]
        elif kind == 'help':
            touched = [r[3:] for r in schedule.get('helped', []) if r[:3] == (0, nq, c)]
        else:
            touched = []         # (collecting: finished rows of the strip, behind their marks)
        for i, col in touched:
            # whose accesses have to be over: the block's owner's, or, where the panel's parts lie, everybody's
            before = {owner[i, col]} if col < 4 else set(owner.values()) if 32 * i + 31 >= row0 else set()
            assert before <= ({w} if not (kind == 'help' and awaits) else set(owner.values()) | {w}), \
                'wave %d in block (%d, %d)' % (w, i, col)


def test_the_kernel_takes_its_schedule_from_the_header():
    with open(os.path.join(CSRC, 'inverse.hip')) as f:
        text = f.read()
    block = text[text.index('void diag_block('):text.index('void potrf_diag_kernel')]
    for name in ('STRIP_ROLES', 'helped_blocks', 'pending_row', 'pending_col', 'PENDING_WAVES', 'PENDING_ROW0',
                 'helper_awaits_pending'):
        assert name in block
    # marked behind the last access, awaited in front of the first one of either way through a helper's blocks
    assert block.index('pending_marks[wave] = 1.f') > block.index('*s = fmaf(-4.f, acc[e], *s)')
    assert block.count('settle();\n        apply(') == 2
