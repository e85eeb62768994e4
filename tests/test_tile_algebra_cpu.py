"""Index algebra of the tiled partition and of the share's owner rule, restated
in numpy from the comments of pakman_plus_amd/csrc/pk_device.hip and checked on
the CPU against what it stands for: keys by prefix, pieces by search, owners
window by window.  The kernels themselves are checked on the GPU
(test_gpu_tiles.py, test_gpu_borders.py)."""
from __future__ import annotations

import numpy as np
import pytest

import rank_util as RU

M32 = (1 << 32) - 1


def _alignbit(hi, lo, sh):
    return (((hi << 32) | lo) >> (sh & 31)) & M32


# ---------------------------------------------------------------------------
# Level 1: digits from the stream of 2-bit fields shifted down by the digit's
# position, 16 (or 32) k-mer ends per thread.


@pytest.mark.parametrize("words,wpt", [(2, 1), (2, 2), (4, 1), (4, 2)])
def test_digit_words(words, wpt):
    """dw holds bits of E so that the digit of the k-mer that ends at byte j lies
    at a place that depends on j alone, at every digit position and width."""
    rng = np.random.default_rng(words * 10 + wpt)
    E = [int(x) for x in rng.integers(0, 1 << 32, words + wpt, dtype=np.uint64)]  # words before, then the thread's
    stream = 0
    for w in E:
        stream = stream << 32 | w
    bits = 32 * words
    for db in (1, 2, 7, 10):
        for dpos in range(0, bits - db + 1):
            q, sh = dpos >> 5, dpos & 31
            dw = []
            for i in range(wpt + 1):
                c = words + wpt - 1 - i
                lo = E[c - q] if c - q >= 0 else 0
                hi = E[c - q - 1] if c - q - 1 >= 0 else 0
                dw.append(_alignbit(hi, lo, sh))
            for j in range(16 * wpt):
                i = wpt - 1 - (j >> 4)
                digit = _alignbit(dw[i + 1], dw[i], 30 - 2 * (j & 15)) & ((1 << db) - 1)
                # the key is the `bits` bits up to and with byte j's field
                key = (stream >> (2 * (16 * wpt - 1 - j))) & ((1 << bits) - 1)
                assert digit == (key >> dpos) & ((1 << db) - 1), (db, dpos, j)


# ---------------------------------------------------------------------------
# Run tables.


class Level:
    """One level's output: the array, and what a reader finds buckets by."""

    def __init__(self, db, KB, fixed, tiles):
        # tiles: list per parent bucket of lists of keys (a tile each), placed
        # one after another from the parent's first place
        nb = 1 << db
        self.db, self.fixed = db, fixed + db
        self.boff, self.tp = [0], [0]
        S, M = [], []
        for parent in tiles:
            nt = len(parent)
            entries = [[None] * nt for _ in range(nb)]
            for t, tile in enumerate(parent):
                d = [(k >> (KB - fixed - db)) & (nb - 1) for k in tile]
                order = sorted(range(len(tile)), key=lambda i: d[i])  # any order inside a digit
                S += [tile[i] for i in order]
                start = 0
                for x in range(nb):
                    c = d.count(x)
                    entries[x][t] = (start, c)
                    start += c
            M += [e for row in entries for e in row]  # (tp[a] << db) + s * ntiles(a) + t
            self.boff.append(self.boff[-1] + sum(len(t) for t in parent))
            self.tp.append(self.tp[-1] + nt)
        self.S, self.M = S, M
        self.V = [0]
        for _, c in M:
            self.V.append(self.V[-1] + c)
        self.tile_len = [[len(t) for t in p] for p in tiles]

    def bucket(self, b):
        """(virtual start, keys) of bucket b through the run table."""
        a, s = b >> self.db, b & ((1 << self.db) - 1)
        nt = self.tp[a + 1] - self.tp[a]
        e0 = (self.tp[a] << self.db) + s * nt
        out = []
        for t in range(nt):
            place = self.boff[a] + sum(self.tile_len[a][:t])
            st, c = self.M[e0 + t]
            out += self.S[place + st:place + st + c]
        return self.V[e0], out


@pytest.mark.parametrize("bits", [(3,), (1, 4), (3, 2, 2)])
def test_run_tables(bits):
    """Buckets read through one, two and three run tables hold the keys with their
    prefix, at virtual places in key order; uneven tiles, empty tiles and digits
    without keys among them."""
    rng = np.random.default_rng(sum(bits))
    KB, N = 16, 700
    keys = [int(k) for k in rng.integers(0, 1 << KB, N)]
    keys[:200] = [k & 0x0FFF | 0x2000 for k in keys[:200]]  # skewed
    cuts = sorted({0, N, 3, 3, *(int(x) for x in rng.integers(0, N, 9))})
    tiles = [[keys[a:b] for a, b in zip(cuts, cuts[1:])] + [[]]]
    fixed, lv = 0, None
    for i, db in enumerate(bits):
        lv = Level(db, KB, fixed, tiles)
        fixed += db
        at = 0
        for b in range(1 << fixed):
            v, got = lv.bucket(b)
            assert v == at
            assert sorted(got) == sorted(k for k in keys if k >> (KB - fixed) == b)
            at += len(got)
        assert at == N and lv.V[-1] == N
        # the next level's tiles: tk keys at a time of every bucket
        tk = 64
        buckets = [lv.bucket(b)[1] for b in range(1 << fixed)]
        tiles = [[x[j:j + tk] for j in range(0, len(x), tk)] for x in buckets]


@pytest.mark.parametrize("seed", range(6))
def test_piece_map(seed):
    """Word bits and counts before a word give a place's piece, pieces without
    places and a first piece that began before the range among them."""
    rng = np.random.default_rng(seed)
    counts = rng.integers(0, 9, 120) * (rng.random(120) < 0.6)
    V = np.concatenate([[0], np.cumsum(counts)])
    v0 = int(rng.integers(0, V[-1] // 2))
    m = int(rng.integers(1, V[-1] - v0 + 1))
    nwords = (m + 31) // 32
    x, y, piece = [0] * nwords, [0] * nwords, []
    for idx in range(120):
        vs, ve = int(V[idx]), int(V[idx + 1])
        if ve > vs and vs < v0 + m and ve > v0:
            ls = max(vs - v0, 0)
            x[ls >> 5] |= 1 << (ls & 31)
            piece.append((idx, vs))
    for w in range(1, nwords):
        y[w] = y[w - 1] + bin(x[w - 1]).count("1")
    for i in range(m):
        low = M32 >> (31 - (i & 31))
        r = y[i >> 5] + bin(x[i >> 5] & low).count("1") - 1
        idx, vs = piece[r]
        want = int(np.searchsorted(V, v0 + i, side="right")) - 1
        assert idx == want, i


# ---------------------------------------------------------------------------
# The owner rule.


def _decided(fa: bytes, k: int, P: int, freq, keep_last_lane=True):
    """[(end byte, owner or None)] of the valid windows as k_own decides them:
    None where an end before the window's last is dirty (the walk follows those),
    except in the first window of a read.  keep_last_lane = False looks for the
    line end after a word in the word itself in lane 63, a planted mistake."""
    n, w = len(fa), k - RU.L + 1
    code = [RU.code3(b) for b in fa] + [0]
    rows = []
    pos = fa.find(b">")
    while 0 <= pos < n:
        q = fa.find(b"\n", pos)
        s = q + 1
        e = fa.find(b"\n", s)
        e = n if e < 0 else e
        exact, back = {}, {}
        for x in range(s + RU.L - 1, e):
            v = 0
            for j in range(RU.L):
                v |= code[x - RU.L + 1 + j] << (2 * (RU.L - 1 - j))
            exact[x] = v & RU.LMASK
            back[x] = (v | code[x + 1] >> 2) & RU.LMASK

        def dirty(x):
            if exact[x] == back[x]:
                return False
            # the last byte of a word: is the next word's first byte a line end?
            lane = (x // 16 % 508 + 4) % 64
            if x % 16 == 15 and lane == 63:
                return True if keep_last_lane else fa[x - 15] != 10
            return not (x + 1 < n and fa[x + 1] == 10)

        for end in range(s + k - 1, e):
            ends = range(end - w + 1, end + 1)
            first = end == s + k - 1
            if not first and any(dirty(x) for x in ends[:-1]):
                rows.append((end, None))
                continue
            best = min(ends, key=lambda x: (int(freq[exact[x]]), x))
            rows.append((end, RU.hash31(exact[best]) % P))
        pos = e + 1
    return rows


def _case(rng, k, word):
    """A line end at a word's first byte and N right after the word, behind A."""
    acgt = np.frombuffer(b"ACGT", dtype=np.uint8)
    last = b">hh\n"
    fill = b"\n" + bytes(rng.choice(acgt, 70)) + b"\n"
    at = 16 * word
    fa = b">" + b"f" * (at + 1 - len(last) - len(fill) - 1) + fill + last
    return fa + bytes(rng.choice(acgt, 14)) + b"AN" + bytes(rng.choice(acgt, 110)) + b"\n"


@pytest.mark.parametrize("k", [9, 31, 64])
def test_owner_rule(k):
    """Windows the rule decides have the owner of the window-by-window walk, with
    the word of the line end in lanes 62, 63 and 0."""
    rng = np.random.default_rng(k)
    for word in (58, 59, 60, 123):
        for _ in range(6):
            fa = _case(rng, k, word)
            freq = RU.lmer_freq(fa)
            walk = [o for _, o in RU.owner_walk(fa, k, 8, freq)]
            rows = _decided(fa, k, 8, freq)
            assert len(rows) == len(walk)
            assert all(o is None or o == w for (_, o), w in zip(rows, walk))


def test_owner_rule_without_the_last_lane():
    """Taking lane 63's next line end from its own word decides windows wrongly,
    and only there."""
    rng = np.random.default_rng(5)
    wrong = {58: 0, 59: 0, 60: 0}
    for word in wrong:
        for _ in range(20):
            fa = _case(rng, 31, word)
            freq = RU.lmer_freq(fa)
            walk = [o for _, o in RU.owner_walk(fa, 31, 8, freq)]
            rows = _decided(fa, 31, 8, freq, keep_last_lane=False)
            wrong[word] += any(o is not None and o != w for (_, o), w in zip(rows, walk))
    assert wrong[58] == 0 and wrong[60] == 0 and wrong[59] > 5
