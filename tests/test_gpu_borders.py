"""Inputs that put the thing a kernel treats specially right at the border of
a wave, a block, a tile or a batch, bit-exact against the oracle or a
restatement."""
from __future__ import annotations

import sys
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _p(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def ctx():
    from pakman_plus_amd import api
    c = api.Context(0)
    yield c
    c.close()


def _bases(rng, n, alpha=b"ACGT"):
    return bytes(rng.choice(np.frombuffer(alpha, dtype=np.uint8), n))


def _shares_match(ctx, fa, k, P):
    """Every rank's share against the window-by-window restatement."""
    import rank_util as RU
    freq = RU.lmer_freq(fa)
    walk = RU.owner_walk(fa, k, P, freq)
    for r in range(P):
        ctx.count_rank_share(fa, k, P, r)
        keys, counts = ctx.table_host()
        assert RU.table_counter(keys, counts) == RU.share_counter(walk, r), r


@pytest.mark.parametrize("k", [9, 15, 31, 64])
@pytest.mark.parametrize("tile", [0, 1])
@pytest.mark.parametrize("ends", ["header", "sequence"])
def test_share_line_end_in_a_waves_last_word(ctx, k, tile, ends):
    """The owner rule takes 16-byte words, 64 a wave and 508 a tile (its first
    wave starts four words before the tile): a line end at the first byte of a
    wave's last word, and of the words on either side of it, and right behind
    that word a byte whose third code bit is set, after a base whose low code
    bit is clear, so that the L-mer that ends there is another one when it is
    read back from the k-mer.  The line end is a header's, or a read's with an
    empty header after it."""
    rng = np.random.default_rng(1000 * k + 10 * tile + len(ends))
    for word in [508 * tile + 64 * wave + lane - 4 for wave in (0, 1, 7) for lane in (62, 63, 64)]:
        at = 16 * word
        for trial in range(8):
            _p(f"case: share line end k={k} tile={tile} {ends} word={word} trial={trial}")
            if ends == "header":
                last, first = b">" + b"h" * 9 + b"\n", _bases(rng, 14)
            else:
                last, first = b">\n" + _bases(rng, 30) + b"\n", b">\n" + _bases(rng, 12)
            fill = b"\n" + _bases(rng, 80) + b"\n"
            fa = b">" + b"f" * (at + 1 - len(last) - len(fill) - 1) + fill + last
            assert len(fa) == at + 1
            fa += first + b"AN" + _bases(rng, 130) + b"\n"
            assert fa[at] == 10 and fa[at + 15:at + 17] == b"AN"
            _shares_match(ctx, fa, k, 3)


@pytest.mark.parametrize("k", [9, 31, 64])
def test_share_of_reads_at_every_alignment(ctx, k):
    """As many records of 131 bytes as a tile has bytes (8128), each with bytes
    outside A, C, G and T among its first bases: every place of a line end in a
    tile occurs."""
    rng = np.random.default_rng(k)
    reads = []
    for i in range(8128):
        r = bytearray(_bases(rng, 128))
        for p in rng.integers(17, 60, 2):
            r[p] = b"NnX"[p % 3]
        r[14:16] = b"AN"
        reads.append(b">\n" + bytes(r) + b"\n")
    assert len(reads[0]) == 131
    _p(f"case: share at every alignment k={k}")
    _shares_match(ctx, b"".join(reads), k, 2)


@pytest.mark.parametrize("k", [24, 32, 33, 40, 64])
def test_bucket_whose_later_batch_has_too_many_runs(ctx, oracle_mod, k):
    """Buckets of several batches: the first keys come from a few tiles, the last
    ones from 900 tiles with two keys each, more runs than a batch's map holds,
    which the first wave finds while the others end the batch before."""
    rng = np.random.default_rng(k)
    genome = _bases(rng, 8_000)

    def cut(n):
        a = int(rng.integers(0, len(genome) - n))
        return genome[a:a + n]

    fa = b"".join(b">a\n" + cut(k + 99) + b"\n" for _ in range(500))
    fa += b"".join(b">" + b"h" * (16_384 - k - 18) + b"\n" + cut(k + 15) + b"\n" for _ in range(900))
    try:
        ctx.set_tuning(l1_bits=10, bucket_factor=10.0)
        _p(f"case: late runs k={k}")
        ctx.count(fa, k)
        keys, counts = ctx.table_host()
    finally:
        ctx.set_tuning()
    want_k, want_c = oracle_mod.count(fa, k)
    assert np.array_equal(keys.reshape(-1), np.asarray(want_k).reshape(-1))
    assert np.array_equal(counts, want_c)


@pytest.mark.parametrize("klen,bits", [(32, 64), (64, 128)])
def test_builder_reads_to_the_end_of_the_input(klen, bits):
    """A million records with a read length beyond the input: their reads run to
    its end, 4e13 windows, which no budget has room for; refused as soon as their
    number is known, and the context counts on."""
    from pakman_plus_amd import api
    rng = np.random.default_rng(klen)
    rows = np.full((1_000_000, 74), 10, dtype=np.uint8)
    rows[:, 0] = ord(">")
    rows[:, 2:73] = rng.choice(np.frombuffer(b"ACGT", dtype=np.uint8), (rows.shape[0], 71))
    fa = rows.tobytes()
    c = api.Context(0, 8 << 30)
    try:
        c.builder_count(fa, klen, read_len=71, kmer_bits=bits)
        want = c.table_host()
        _p(f"case: reads to the end klen={klen}")
        t = time.perf_counter()
        with pytest.raises(api.PakHipError) as e:
            c.builder_count(fa, klen, read_len=0xFFFFFFF0, kmer_bits=bits)
        assert e.value.code == api.PK_ENOMEM
        assert time.perf_counter() - t < 5.0
        assert c.builder_count(fa, klen, read_len=71, kmer_bits=bits) == rows.shape[0]
        got = c.table_host()
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    finally:
        c.close()


@pytest.mark.parametrize("run", [1, 14, 15, 16, 17, 31, 33, 1_023, 1_024, 1_025, 70_000])
@pytest.mark.parametrize("end", [b"\n", b"\r\n"])
def test_rewrite_over_blank_lines(ctx, oracle_mod, run, end):
    """Runs of blank lines between a read's lines, after it, before the first
    record and at the input's end, shorter and longer than a chunk steps over one
    by one and than a block's table holds."""
    rng = np.random.default_rng(run)
    n = max(3, min(400, 150_000 // run))
    parts = [end * run]
    for i in range(n):
        parts += [b">%d" % i + end]
        for _ in range(int(rng.integers(0, 4))):
            parts += [_bases(rng, int(rng.integers(1, 40)), b"ACGTN") + end, end * int(rng.integers(0, 2)) * run]
    fa = b"".join(parts) + end * run
    _p(f"case: blank lines run={run} end={end!r}")
    assert ctx.normalize(fa, "fasta") == oracle_mod.normalize(fa, "fasta")


def test_rewrite_time_over_blank_lines(ctx):
    """A run of four million blank lines takes about as long as as many lines of
    one base (0.5 ms; stepped over by one thread 0.8 s)."""
    read = b">r\n" + b"ACGT" * 25 + b"\n"
    _p("case: time over blank lines")
    for _ in range(2):
        ctx.normalize(read + b"\n" * 4_000_000 + read, "fasta")
    assert ctx.timing()["normalize_ms"] < 20.0


def test_split_of_buckets_with_many_runs(ctx, oracle_mod):
    """Words that reach back to the read's start, short at first: a few buckets
    hold a good part of the keys, in runs of every tile, and go through the split.
    It takes 3.4 ms (13.5 with one block gathering each bucket's runs)."""
    rng = np.random.default_rng(2)
    genome = np.frombuffer(_bases(rng, 2_000_000), dtype=np.uint8)
    at = rng.integers(0, genome.size - 100, 400_000)
    rows = np.full((at.size, 104), 10, dtype=np.uint8)
    rows[:, :3] = np.frombuffer(b">r\n", dtype=np.uint8)
    rows[:, 3:103] = genome[at[:, None] + np.arange(100)]
    for reads in (30_000, at.size):
        fa = rows[:reads].tobytes()
        _p(f"case: split of buckets with many runs reads={reads}")
        for _ in range(3):
            n = ctx.builder_count(fa, 11, read_len=100, kmer_bits=64)
        t = ctx.timing()
        keys, counts = ctx.table_host()
        keys = keys.reshape(-1)
        assert n == reads and t["n_split"] > 0
        if reads < at.size:
            want_n, want_k, want_c = oracle_mod.builder_count(fa, 11, 100, 64)
            assert n == want_n
            assert np.array_equal(keys, np.asarray(want_k).reshape(-1)) and np.array_equal(counts, want_c)
    assert np.all(keys[1:] > keys[:-1]) and int(counts.sum()) == 90 * reads
    assert t["split_ms"] < 8.0


@pytest.mark.parametrize("k", [32, 64])
def test_bucket_of_equal_keys(ctx, oracle_mod, k):
    """Most k-mers of the input equal, the others in the same bucket and beside
    it: one block counts them, in one pass (1e7 of k = 32: 23 ms; in sixteen passes
    137)."""
    rng = np.random.default_rng(k)
    tail = b"".join(b">t\n" + b"A" * (k // 2) + _bases(rng, 2 * k) + b"\n" for _ in range(50))
    read = b">r\n" + b"A" * 150 + b"\n"
    n = 10_000_000 // (151 - k)
    _p(f"case: equal keys k={k}")
    for _ in range(2):
        ctx.count(read * n + tail, k)
    keys, counts = ctx.table_host()
    want_k, want_c = oracle_mod.count(read + tail, k)
    want_c = np.array(want_c)
    want_c[0] += (n - 1) * (151 - k)  # A is 0: the first key
    assert np.array_equal(keys.reshape(-1), np.asarray(want_k).reshape(-1))
    assert np.array_equal(counts, want_c)
    assert ctx.timing()["sort_ms"] < 60.0


@pytest.mark.parametrize("k", [32, 40])
def test_retry_of_few_buckets_among_a_million(ctx, oracle_mod, k):
    """2^20 buckets, nearly all of one or two keys, and a few with more distinct
    keys than a table holds, up to the very last one: each is found and counted
    in several passes, with more and with fewer keys than a batch."""
    rng = np.random.default_rng(k)
    acgt = np.frombuffer(b"ACGT", dtype=np.uint8)
    some = rng.choice(acgt, (1_200_000, k))
    groups = [some]
    for prefix, n in ((b"A" * 10, 3_000), (b"ACGTACGTAC", 7_000), (b"T" * 10, 4_000), (b"G" * 9 + b"T", 2_700),
                      (b"G" * 10, 30_000)):
        g = rng.choice(acgt, (n, k))
        g[:, :10] = np.frombuffer(prefix, dtype=np.uint8)
        groups.append(g)
    reads = np.concatenate(groups)
    rows = np.full((reads.shape[0], k + 4), 10, dtype=np.uint8)
    rows[:, :3] = np.frombuffer(b">r\n", dtype=np.uint8)
    rows[:, 3:-1] = reads[rng.permutation(reads.shape[0])]
    fa = rows.tobytes()
    try:
        ctx.set_tuning(bucket_factor=1.2 / (1920 if k <= 32 else 1152))  # one instance a bucket
        _p(f"case: retry among a million buckets k={k}")
        ctx.count(fa, k)
        assert ctx.timing()["bucket_bits"] == 20
        keys, counts = ctx.table_host()
    finally:
        ctx.set_tuning()
    want_k, want_c = oracle_mod.count(fa, k)
    assert np.array_equal(keys.reshape(-1), np.asarray(want_k).reshape(-1))
    assert np.array_equal(counts, want_c)


def test_time_of_distinct_keys(ctx):
    """6.9e7 k-mers, all distinct: every bucket's first table is too small.  The
    bucket count takes 1.8 ms (5.6 with the pass that had failed repeated and the
    keys loaded again for each pass)."""
    rng = np.random.default_rng(3)
    rows = np.full((1_000_000, 104), 10, dtype=np.uint8)
    rows[:, :3] = np.frombuffer(b">r\n", dtype=np.uint8)
    rows[:, 3:103] = rng.choice(np.frombuffer(b"ACGT", dtype=np.uint8), (rows.shape[0], 100))
    fa = rows.tobytes()
    _p("case: time of distinct keys")
    for _ in range(3):
        n = ctx.count(fa, 32).n
    keys, counts = ctx.table_host()
    assert np.all(keys[1:, 0] > keys[:-1, 0]) and n > 68_900_000 and int(counts.sum()) == 69_000_000
    assert ctx.timing()["sort_ms"] < 3.6


@pytest.mark.parametrize("k", [32, 50])
@pytest.mark.parametrize("l1_bits,further", [(10, 0), (7, 1), (5, 1), (3, 2), (2, 2)])
def test_partition_levels(ctx, oracle_mod, k, l1_bits, further):
    """One, two and three partition levels over the same reads, ragged tiles and
    empty digits among them."""
    rng = np.random.default_rng(9)
    genome = _bases(rng, 60_000)
    fa = b"".join(b">r%d\n" % i + genome[a:a + 60 + i % 90] + b"\n"
                  for i, a in enumerate(rng.integers(0, 59_800, 12_000).tolist()))
    bits = 10 if further == 0 else 14
    n = sum(max(60 + i % 90 - k + 1, 0) for i in range(12_000))
    cap = 1920 if k <= 32 else 1152
    try:
        # a factor that gives a bucket its share of n at that many bits
        ctx.set_tuning(l1_bits=l1_bits, bucket_factor=1.01 * (n >> bits) / cap)
        _p(f"case: levels k={k} l1_bits={l1_bits}")
        ctx.count(fa, k)
        t = ctx.timing()
        assert (t["bucket_bits"], t["ms_levels"]) == (bits, further)
        keys, counts = ctx.table_host()
    finally:
        ctx.set_tuning()
    want_k, want_c = oracle_mod.count(fa, k)
    assert np.array_equal(keys.reshape(-1), np.asarray(want_k).reshape(-1))
    assert np.array_equal(counts, want_c)
