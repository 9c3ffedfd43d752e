"""CPU: runs cut at multiples of a piece of several work-groups' entries, and the order in which the work-groups of the
entry-parallel kernels take their segments (smm_mfma.hip), emulated step by step."""
import numpy as np

from tests.test_cut_rules import check, cut, stacks

CUS, MOST = 256, 2048


def segment(w, groups, spread):
    """the segment of work-group w of groups"""
    if not spread or groups <= CUS or MOST < groups:
        return w
    x, share = w % CUS, groups // CUS
    return x * share + min(x, groups % CUS) + w // CUS


def test_every_segment_once():
    for groups in list(range(1, 600, 7)) + [255, 256, 257, 511, 512, 513, 2047, 2048, 2049, 4095]:
        assert sorted(segment(w, groups, True) for w in range(groups)) == list(range(groups))
    for groups in (300, 1000, 2048):  # neighbours meet on one CU: w, w + 256, ..
        for x in range(0, CUS, 17):
            mine = [segment(w, groups, True) for w in range(x, groups, CUS)]
            assert mine == list(range(mine[0], mine[0] + len(mine)))


def walk(c, seg, bs, piece, T):
    """the pieces of one work-group: ep_body's head search and run ends"""
    S = len(c)
    begin, end = seg * bs, min(seg * bs + bs, S)
    h = next((x for x in range(begin, end) if x == 0 or c[x] != c[x - 1] or
              (x == begin and 0 == x % piece and cut(c, x, c[x], T))), end)
    pieces = []
    while h < end:
        c0, r = c[h], h + 1
        while r < S and not (c[r] != c0 or (end <= r and 0 == r % piece and cut(c, r, c0, T))):
            r += 1
        pieces.append((c0, list(range(h, r)), (h > 0 and c[h - 1] == c0) or (r < S and c[r] == c0)))
        h = r
    return pieces


def test_pieces_exactly_once():
    rng = np.random.default_rng(4)
    for c, srt in stacks(rng, 1500):
        bs = int(rng.integers(1, 20))
        piece, T = bs * int(rng.integers(1, 6)), int(rng.integers(0, 60))
        groups = (len(c) + bs - 1) // bs
        check(c, [p for w in range(groups) for p in walk(c, segment(w, groups, True), bs, piece, T)], srt)


def test_long_run_in_pieces():
    """a run far longer than T: pieces of about the given length whatever the work-group's entries"""
    c = np.zeros(3000, dtype=int)
    for bs, piece, T in ((2, 8, 12), (8, 24, 40), (5, 15, 15)):
        lengths = [len(p[1]) for w in range((3000 + bs - 1) // bs) for p in walk(c, w, bs, piece, T)]
        assert sum(lengths) == 3000 and max(lengths) <= T + piece + bs and sorted(lengths)[len(lengths) // 2] == piece
